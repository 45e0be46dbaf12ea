"""The engine's host-side bound of its positions, which sizes the prefill's
attention: kept through reset / step / prefill, given up (max_len 0, the cache's
capacity) as soon as positions may change without the host.  On the CPU, with
recording stand-ins for the kernels."""
import contextlib
import importlib.util
import os
import types

import pytest

torch = pytest.importorskip("torch")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _engine_mod():
    spec = importlib.util.spec_from_file_location("qw_engine", os.path.join(ROOT, "qwen3.5_0.8b_deploy_amd", "engine.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


@pytest.fixture
def make():
    em = _engine_mod()
    em._capturing = lambda stream: stream == "capturing"
    calls = []
    names = ("embedding_gather", "rmsnorm", "linear", "mlp_fused", "layer_tail", "lmhead_argmax")
    qw = types.SimpleNamespace(**{n: lambda *a, **k: None for n in names})
    qw.attn_forward = lambda *a, tokens, max_len, **k: calls.append((tokens, max_len))
    qw.positions_add = lambda ctx, pos, n, stream=None: pos.add_(n)

    def engine(B=2, capacity=1000):
        e = em.DecodeEngine.__new__(em.DecodeEngine)
        e.qw, e.ctx, e.B, e.capacity, e.act, e.norm_first = qw, None, B, capacity, torch.float32, False
        e.layers = [dict.fromkeys(("in_norm", "post_norm", "in", "out", "gateup", "down", "q_norm", "k_norm", "E"))]
        e.layers[0].update(linear=False, cache=(torch.zeros(1),))
        e.embed = e.E = e.final_norm = None
        e.x = e.xn = torch.zeros(B, em.H)
        e.row, e.core = torch.zeros(B, em.FULL_IN), torch.zeros(B, em.FNH * em.HD)
        e.ids = torch.zeros(B, dtype=torch.int32)
        e._pos, e._end, e._shared = torch.zeros(B, dtype=torch.int32), 0, False
        e.check = lambda: None
        return e, calls
    return engine


def ids(T, B=2):
    return torch.zeros(B, T, dtype=torch.int32)


@pytest.mark.parametrize("stream", [None, "a stream"])
def test_prefill_is_sized_by_the_positions(make, monkeypatch, stream):
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    e, calls = make()
    e.reset([1, 2])
    e.prefill(ids(100), stream=stream)
    e.step(stream=stream)
    e.prefill(ids(30), stream=stream)
    e.reset([1, 2], [5, 400])
    e.prefill(ids(64), stream=stream)
    assert calls == [(100, 100), (1, 1000), (30, 131), (64, 464)]


def test_bound_stays_inside_the_cache(make):
    e, calls = make()
    e.reset([1, 2], torch.tensor([990, 3]))
    e.prefill(ids(64))
    e.reset([1, 2], [-500, -500])
    e.prefill(ids(16))
    assert calls == [(64, 1000), (16, 1)]


def test_unseen_changes_give_the_bound_up(make):
    """A captured step (before or after a reset), the tensor handed out or replaced."""
    for unseen in (lambda e: e.step(stream="capturing"), lambda e: e.pos, lambda e: setattr(e, "pos", e._pos.clone())):
        for first in (True, False):
            e, calls = make()
            del calls[:]
            if first:
                unseen(e)
            e.reset([1, 2])
            if not first:
                unseen(e)
            e.prefill(ids(50))
            e.reset([1, 2])  # a graph may be replayed after it all the same
            e.prefill(ids(50))
            assert [c for c in calls if c[0] == 50] == [(50, 0), (50, 0)]


def test_captured_step_is_seen_while_the_bound_is_not_known(make):
    e, calls = make()
    e._end = None  # as after positions that were on the device
    e.step(stream="capturing")
    e.reset([1, 2])
    e.prefill(ids(50))
    assert calls[-1] == (50, 0)
