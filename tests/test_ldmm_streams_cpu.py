"""The two-stream form of ldmm joins its side stream on every way out (streams and launches are recorded, not run)."""
import contextlib
import importlib

import pytest
import torch

ldmm_module = importlib.import_module("triteia_amd.python.ops.matmul.ldmm")


class _Stream:
    def __init__(self, name, events):
        self.name, self.events = name, events

    def wait_stream(self, other):
        self.events.append(f"{self.name} waits for {other.name}")


@pytest.mark.parametrize("deltas", [0, 2])
@pytest.mark.parametrize("failing", [None, "plan", "shrink", "expand", "delta"])
def test_side_stream_is_joined(monkeypatch, failing, deltas):
    events = []
    cur, side = _Stream("current", events), _Stream("side", events)
    on = [cur]

    @contextlib.contextmanager
    def stream(s):
        on.append(s)
        yield
        on.pop()

    def step(name):
        def run(*args, **kwargs):
            what = name if name != "sgmv" else "shrink" if kwargs.get("accumulate") is False else "expand"
            events.append(f"{what} on {on[-1].name}")
            if what == failing:
                raise RuntimeError("refused")
        return run

    class Declines:
        def ldmm(self, *args):
            return None

    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: cur)
    monkeypatch.setattr(torch.cuda, "stream", stream)
    monkeypatch.setattr(ldmm_module, "_side_stream", lambda device: side)
    monkeypatch.setattr(ldmm_module, "native", Declines)
    monkeypatch.setattr(ldmm_module, "routed_workspace", lambda *args: None)
    for name, what in (("route_plan", "plan"), ("sgmv_routed", "sgmv"), ("sbmm_2_4_routed", "delta")):
        monkeypatch.setattr(ldmm_module, name, step(what))
    x = torch.zeros(4, 64, dtype=torch.float16)
    A, B = torch.zeros(3, 64, 8, dtype=torch.float16), torch.zeros(3, 8, 128, dtype=torch.float16)
    q = torch.zeros(deltas, 2, 256, dtype=torch.int32)
    base = torch.zeros(128, 64, dtype=torch.float16)
    call = lambda: ldmm_module.ldmm(torch.zeros(4, dtype=torch.int32), x, A, B, q, None, None, base_weight=base)
    if failing is None or (failing == "delta" and deltas == 0):
        call()
    else:
        with pytest.raises(RuntimeError, match="refused"):
            call()
    work = [i for i, e in enumerate(events) if e.endswith("on side")]
    assert work and max(work) < max(i for i, e in enumerate(events) if e == "current waits for side")
