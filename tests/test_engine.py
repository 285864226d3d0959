"""CPU tests of Engine's staging and launches: which calls a staged step makes, with the launches
recorded instead of issued."""
import contextlib
import types

import numpy as np
import pytest
import torch

F16, BF16, FP8 = 1, 2, 3
LAUNCHES = ("attention_plan", "kv_append", "attention_partial", "attention_partial_append",
            "attention_partial_append_fp8", "attention_merge", "paged_attention")


@pytest.fixture
def engine(lia, monkeypatch):
    """engine(kv_dtype) -> an Engine on host memory that records its launches."""
    calls, used = [], set()
    for name in LAUNCHES:
        def record(*a, _name=name, **k):
            calls.append(_name)
            used.update(t.data_ptr() for t in a if isinstance(t, torch.Tensor))

        monkeypatch.setattr(lia, name, record)
    stream = types.SimpleNamespace(cuda_stream=0, synchronize=lambda: calls.append("synchronize"))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: stream)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)

    @contextlib.contextmanager
    def device(d):
        calls.append(f"device {d}")
        yield
        calls.append("device back")

    monkeypatch.setattr(torch.cuda, "device", device)
    zeros = torch.zeros
    monkeypatch.setattr(torch, "zeros", lambda *a, pin_memory=False, **k: zeros(*a, **k))

    def make(kv_dtype=F16, maximum_sequences=4):
        e = lia.Engine(16, 2, 128, pool_tokens=2048, layers=1, page_size=32, kv_dtype=kv_dtype,
                       prefill_batch=64, device="cpu")
        e.configure_paging(maximum_sequences, 1024)
        e.calls, e.used = calls, used  # names of the launches, addresses of their tensors
        return e

    return make


def attend(e, n, dtype):
    """The launches of one layer of the staged step on rows of `dtype`."""
    del e.calls[:]
    rows = torch.zeros((n, 2, 128), dtype=dtype)
    e.attention(0, torch.zeros((n, 16, 128)), rows, rows)
    return list(e.calls)


INTERLEAVED = [(1, 100, 0), (1, 500, 1), (1, 101, 0)], [list(range(4)), list(range(4, 20))]
SHARED = [(1, 40, 0), (1, 64, 1)], [[2, 3], [5, 3, 6]]  # sequence 1 attends page 3, sequence 0 writes it
PRIVATE = [(1, 100, 0), (1, 101, 0), (1, 500, 1)], [list(range(4)), list(range(4, 20))]


@pytest.mark.parametrize("kv,dtype", [(F16, torch.float16), (BF16, torch.bfloat16)])
@pytest.mark.parametrize("batch,fused", [(INTERLEAVED, False), (SHARED, False), (PRIVATE, True)])
def test_rows_that_the_step_itself_attends_are_appended_first(engine, kv, dtype, batch, fused):
    """The attention launch appends the rows only where it reads no cached key from a slot it writes."""
    e = engine(kv)
    e.stage(*batch)
    want = ["attention_partial_append"] if fused else ["kv_append", "attention_partial"]
    assert attend(e, len(batch[0]), dtype) == want + ["attention_merge"]


def test_append_fusable_equals_a_search_of_every_cached_key(lia):
    """lia_append_fusable against the definition, on batches with shared, repeated and private pages."""
    rng = np.random.default_rng(3)
    P, pool, context = 16, 24, 160
    lim = lia.PagingLimits(4, context, P, pool, 10, 64)
    seen = set()
    for _ in range(400):
        tables = [[int(x) for x in rng.integers(0, pool, 10)] if rng.random() < 0.5
                  else [int(x) for x in rng.permutation(pool)[:10]] for _ in range(4)]
        rows = []
        for s in range(int(rng.integers(1, 5))):
            p0 = int(rng.choice([0, 15, 16, 17, *rng.integers(0, 150, 3)]))
            rows += [(1, p, s) for p in range(p0, min(context, p0 + int(rng.integers(1, 5))))]
        if rng.random() < 0.4:
            rows.sort(key=lambda r: (r[1] % 2, r[2], r[1]))
        try:
            got = lia.pack_rows(lim, rows, tables)
        except lia.LiaError:
            continue
        cu = got["cu_seqlens"]
        args = [np.ascontiguousarray(got[k]) for k in ("positions", "sequences", "flat", "cu_seqlens", "slot_mapping")]
        fusable = lia.lib().lia_append_fusable(lim, len(rows), len(cu) - 1, *[a.ctypes.data for a in args])
        read = {tables[rows[r][2]][p // P] * P + p % P for r in cu[:-1] for p in range(rows[r][1])}
        assert fusable == (not read & set(got["slot_mapping"].tolist()))
        seen.add(fusable)
    assert seen == {0, 1}


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_a_staged_plan_lies_apart_from_the_callers_workspace(engine, dtype):
    """paging["workspace"] may serve other calls between stage() and the last layer."""
    e = engine()
    e.stage(*PRIVATE)
    attend(e, 3, dtype)
    assert e._step_workspace.data_ptr() in e.used and e.paging["workspace"].data_ptr() not in e.used


def test_a_captured_layer_plans_and_appends_for_itself(engine, monkeypatch):
    """The graph of a layer is replayed for later steps, which may attend rows that they append."""
    e = engine()
    e.stage(*PRIVATE)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert attend(e, 3, torch.float16) == ["kv_append", "paged_attention"]


def test_stage_works_on_the_pools_device(engine):
    """The plan is launched where the pool lies, whichever device is current."""
    e = engine()
    e.stage(*PRIVATE)
    assert e.calls == ["device cpu", "attention_plan", "synchronize", "device back"]


def test_an_interrupted_stage_ends_its_copy(engine, lia, monkeypatch):
    """The next stage() writes the pinned image that the copy reads."""
    e = engine()

    def interrupted(*a):
        raise KeyboardInterrupt

    monkeypatch.setattr(lia, "attention_plan", interrupted)
    with pytest.raises(KeyboardInterrupt):
        e.stage(*PRIVATE)
    assert "synchronize" in e.calls
