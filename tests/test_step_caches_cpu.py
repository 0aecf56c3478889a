"""What a head step enqueues, and on what: it returns while its backward is still enqueued, so a call on another stream that shares its caches has to be ordered
behind it.  The launches are replaced by a log here; the streams and events are names."""
import pytest
import torch

from chatlearn_amd import fused, ops


class _Stream:
    device = torch.device("cpu")

    def __init__(self, name, log):
        self.name, self.log, self.cuda_stream = name, log, 0 if name == "default" else id(name)

    def wait_event(self, event):
        self.log.append(("wait", self.name, event.at))

    def record_event(self):
        event = torch.cuda.Event()
        event.record(self)
        return event


@pytest.fixture
def on(monkeypatch):
    """``on(stream, caches...)`` runs a step on that stream; ``on.log`` is what happened, in order."""
    log, state = [], {"stream": None, "capturing": False, "fail": False}

    class Event:
        at = None

        def record(self, stream):
            self.at = sum(1 for e in log if e[0] == "enqueue" and e[1] == stream.name)     # launches of its stream it is behind
            log.append(("record", stream.name, self.at))

    class Step:
        def __init__(self, *a, **kw):
            pass

        def enqueue(self, stages, **kw):
            log.append(("enqueue", state["stream"].name, stages))
            if state["fail"] and stages & 4:
                raise RuntimeError("refused")

    class Flags:
        def __init__(self, values, stream):
            pass

        def tolist(self):
            return [0.0, 3.0]

    streams = {}
    monkeypatch.setattr(ops, "_dev", lambda t, *a: t)
    monkeypatch.setattr(ops, "HeadStep", Step)
    monkeypatch.setattr(fused, "_ReadBack", Flags)
    monkeypatch.setattr(ops, "upload", lambda t, device: t)
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: state["stream"])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda t, s: log.append(("lifetime", s.name, t.data_ptr())))

    def run(name, T=3, capturing=False, fail=False, loss_mask=None, **caches):
        state.update(stream=streams.setdefault(name, _Stream(name, log)), capturing=capturing, fail=fail)
        return fused.grpo_head_step(torch.zeros(T, 64), torch.zeros(5, 64), torch.zeros(T, dtype=torch.int64), torch.zeros(T), None,
                                    torch.zeros(1), torch.tensor([0, T], dtype=torch.int32), loss_mask, n_tokens_total=3.0, **caches)

    run.log = log
    return run


def _launches(log, name):
    return sum(1 for e in log if e[0] == "enqueue" and e[1] == name)


@pytest.mark.parametrize("which", ["workspace_cache", "weight_t_cache"])
@pytest.mark.parametrize("first", ["a", "default"])
def test_another_stream_waits_for_everything_the_last_call_enqueued(on, which, first):
    cache = {}
    on(first, **{which: cache})
    n = _launches(on.log, first)
    on("b", **{which: cache})
    first_b = on.log.index(next(e for e in on.log if e[:2] == ("enqueue", "b")))
    assert ("wait", "b", n) in on.log[:first_b]
    assert cache and all(isinstance(t, torch.Tensor) for t in cache.values())
    shared = [t.data_ptr() for t in cache.values()]
    assert {("lifetime", "b", p) for p in shared} <= set(on.log[:first_b])
    on(first, **{which: cache})
    assert ("wait", first, _launches(on.log, "b")) in on.log


def test_one_stream_waits_for_nothing(on):
    cache, wt = {}, {}
    for name, marks in (("default", 0), ("a", 3)):
        before = len(on.log)
        for _ in range(3):
            on(name, workspace_cache=cache, weight_t_cache=wt)
        assert not any(e[0] in ("wait", "lifetime") for e in on.log[before:])
        assert sum(e[0] == "record" for e in on.log[before:]) == marks
        cache, wt = {}, {}


def test_no_cache_no_event(on):
    on("a")
    on("b")
    assert not any(e[0] in ("wait", "record") for e in on.log)


def test_a_call_that_fails_behind_its_first_launches_is_waited_for(on):
    cache = {}
    with pytest.raises(RuntimeError, match="refused"):
        on("a", fail=True, workspace_cache=cache)
    on("b", workspace_cache=cache)
    assert ("wait", "b", _launches(on.log, "a")) in on.log


def test_capture_neither_waits_nor_leaves_an_event(on):
    """A capture may not depend on work outside of it, nor the reverse: replays are ordered by who replays them."""
    cache = {}
    on("a", workspace_cache=cache)
    before = len(on.log)
    on("b", capturing=True, workspace_cache=cache)
    assert not any(e[0] in ("wait", "record") for e in on.log[before:])
    on("c", workspace_cache=cache)
    assert ("wait", "c", _launches(on.log, "a")) in on.log


@pytest.mark.parametrize("skip_forward,stages", [(True, [1 | 2 | 8, 4 | 8]), (False, [1 | 2, 4])])
def test_the_two_calls_of_a_checked_step_clear_masked_rows_in_one_launch(on, skip_forward, stages):
    """The forward's call has such a launch only where it leaves those rows out."""
    on("a", loss_mask=torch.tensor([1, 0, 1], dtype=torch.int32), skip_masked_forward=skip_forward)
    assert [e[2] for e in on.log if e[0] == "enqueue"] == stages
