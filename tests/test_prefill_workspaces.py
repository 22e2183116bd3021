"""The host side of prompt passes (qwen3/prefill.py, hybrid/prefill.py) on the CPU.

Workspaces: kernels take them as raw pointers with the pass's rows, so a pass must
never find buffers of fewer rows than it was promised.  Dispatch: which prompts of the
hybrids go through a pass and which through the decode step."""
from types import SimpleNamespace

import pytest
import torch

from tilefoundry_amd.hybrid import prefill as hybrid
from tilefoundry_amd.hybrid.prefill import GranitePass, Qwen35Pass
from tilefoundry_amd.qwen3 import prefill as qwen3
from tilefoundry_amd.qwen3.prefill import Prefill

LIB = SimpleNamespace(tfd_panel_gemm_slices=lambda M, K, N: 2)


def _qwen3():
    p = Prefill.__new__(Prefill)
    p.dev, p._lib, p.rows = "cpu", LIB, 0
    p.H, p.QD, p.I, p.qkv_n = 64, 64, 128, 128
    return p, lambda R: {"hid": R * p.H, "h1": R * p.H, "xn": R * p.H, "q": R * p.QD,
                         "attn": R * p.QD, "hmid": R * p.I, "part": 2 * R * 2 * p.I}


def _hybrid(cls):
    p = cls.__new__(cls)
    c = p.cfg = SimpleNamespace(experts=8, shared_inter=64, attn_in=128, moe_inter=32, key_dim=16,
                                value_dim=32, lin_value_heads=2, heads=2, d_inner=64, d_state=16,
                                mamba_heads=2)
    p.dev, p._lib, p.rows, p.H, p.k, p.B = "cpu", LIB, 0, 64, 2, 1
    p.in_rows, p.out_k, p.attn_k = 160, 64, 64

    def sizes(R):
        want = {"emb": R * p.H, "xm": R * p.H, "xn": R * p.H, "stream": R * p.H,
                "part": 2 * R * p.in_rows, "proj": R * p.nproj, "mix": R * p.out_k,
                "rlog": R * c.experts, "rw": R * p.k, "ridx": R * p.k,
                "moe_hidden": R * p.k * c.moe_inter, "d": R * p.k * p.H,
                "shared": R * c.shared_inter, "q": R * p.attn_k}
        if cls is Qwen35Pass:
            want |= {"qk": 2 * R * c.key_dim, "v": R * c.value_dim, "read": R * c.value_dim,
                     "gates": R * c.lin_value_heads * 2, "gate": R * p.attn_k,
                     "self_scores": R * c.heads}
        else:
            want |= {"x": R * c.d_inner, "y": R * c.d_inner, "bc": 2 * R * c.d_state,
                     "gates": R * c.mamba_heads * 2}
        return want

    return p, sizes


PASSES = pytest.mark.parametrize("make", [_qwen3, lambda: _hybrid(Qwen35Pass),
                                          lambda: _hybrid(GranitePass)],
                                 ids=["qwen3", "qwen3_5", "granite"])


@pytest.fixture
def waits(monkeypatch):
    """Called in the place of a wait for the device's current stream."""
    calls = []
    for m in (qwen3, hybrid):
        monkeypatch.setattr(m, "wait_for_work", lambda device: [f() for f in calls])
    return calls


@PASSES
def test_a_failed_growth_promises_nothing(monkeypatch, waits, make):
    """Growing fails at each of its allocations in turn (out of memory, caught by the
    caller): the next pass of the larger size still finds every buffer large enough."""
    real = {n: getattr(torch, n) for n in ("empty", "zeros")}
    left = [0]

    def allocate(name):
        def call(*a, **kw):
            left[0] -= 1
            if left[0] == 0:
                raise torch.OutOfMemoryError("no memory left")
            return real[name](*a, **kw)
        return call

    for n in real:
        monkeypatch.setattr(torch, n, allocate(n))
    for fails_at in range(1, 40):
        p, sizes = make()
        left[0] = 0
        p._reserve(32)
        left[0] = fails_at
        try:
            p._reserve(96)
        except torch.OutOfMemoryError:
            left[0] = 0
            for M in (64, 96):
                p._reserve(M)
                for name, n in sizes(M).items():
                    assert getattr(p, name).numel() >= n, (fails_at, M, name)
        else:
            break
    assert fails_at > 5


@PASSES
def test_buffers_in_use_go_after_a_wait(waits, make):
    """Growing drops buffers that a pass on this stream may still read: it waits once,
    with all of them in place; a first pass and one that fits wait for nothing."""
    p, sizes = make()
    seen = []
    waits.append(lambda: seen.append({n: getattr(p, n).data_ptr() for n in before}))
    before = {}
    p._reserve(32)
    p._reserve(17)
    assert not seen
    before = {n: getattr(p, n).data_ptr() for n in sizes(32)}
    p._reserve(96)
    assert seen == [before]


def _prefilled(monkeypatch, cls, rows, n, routes=None):
    """A prefill of *rows* prompts of *n* tokens on an engine whose sizes a pass takes ->
    (positions walked, whether a pass object was built)."""
    walked, built = [], []
    monkeypatch.setattr(cls, "__init__", lambda self, eng: built.append(eng))
    monkeypatch.setattr(cls, "takes", staticmethod(lambda eng: True))
    monkeypatch.setattr(cls, "run", lambda self, prompts: None)
    monkeypatch.setattr(hybrid, "ptr", lambda t: None)
    z = torch.zeros(rows, dtype=torch.int64)
    eng = SimpleNamespace(B=rows, nsteps=16, replay=lambda: walked.append(1), pos=z.clone(),
                          ids=z.clone(), embed=z, emb=z, err=z, _stream=lambda: 0,
                          cfg=SimpleNamespace(hidden=8, vocab=16), routes=routes,
                          _load_prompts=lambda prompts: None,
                          _lib=SimpleNamespace(tfd_embed_rows_bf16=lambda *a: None))
    hybrid.prefill(eng, cls, [list(range(1, n + 1)) for _ in range(rows)])
    return len(walked), bool(built)


@pytest.mark.parametrize("cls", [Qwen35Pass, GranitePass])
@pytest.mark.parametrize("rows", [1, 2, 16])
def test_a_walked_prompt_builds_no_pass(monkeypatch, cls, rows):
    """One position is walked: nothing is packed or kept for it."""
    assert _prefilled(monkeypatch, cls, rows, 1) == (0, False)
    assert _prefilled(monkeypatch, cls, rows, 2) == (1, False)
    assert _prefilled(monkeypatch, cls, rows, 4) == (0, True)


def test_two_positions_of_one_qwen3_5_sequence_are_walked(monkeypatch):
    """A pass over them is slower than two steps; Granite's, and more sequences', is not."""
    assert _prefilled(monkeypatch, Qwen35Pass, 1, 3) == (2, False)
    assert _prefilled(monkeypatch, Qwen35Pass, 2, 3) == (0, True)
    assert _prefilled(monkeypatch, GranitePass, 1, 3) == (0, True)


@pytest.mark.parametrize("cls", [Qwen35Pass, GranitePass])
def test_an_engine_that_records_routes_is_walked(monkeypatch, cls):
    """``record_routes`` engines hold the experts of the last position walked: a pass has
    none to leave."""
    assert _prefilled(monkeypatch, cls, 2, 9, routes=torch.zeros(1)) == (8, False)
