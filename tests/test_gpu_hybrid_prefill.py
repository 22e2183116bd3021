"""The hybrids' prompt passes (hybrid/prefill.py, csrc/prefill_hybrid.hip) against the
walk of the same prompts through the decode step, on the GPU: caches, recurrent
states, convolution windows and the next step's logits.

Every expert is picked (top_k == experts), so no near-tie of the router decides
anything; the two differ by f32 summation orders, i.e. by roundings to bf16 that
settle the other way.  A value that went through L layers carries at most six rounded
products a layer (in- and out-projection, gate, up, down, the mixer's input), each
2^-9 of it and independent, on both sides: sqrt(2 * 6 L) 2^-9 in the 2-norm, 1.5e-2
for the five layers here; the bound is 2e-2."""
import pytest
import torch

from tilefoundry_amd import _lib
from tilefoundry_amd.hybrid import granite as G
from tilefoundry_amd.hybrid import prefill as P
from tilefoundry_amd.hybrid import qwen3_5 as Q


def test_panel_structs_match_c_layout(tmp_path, monkeypatch):
    from tests import test_abi

    monkeypatch.setattr(test_abi, "STRUCTS", {n: getattr(_lib, n) for n in (
        "TfdPanelMixArgs", "TfdPanelMoeArgs", "TfdPanelGdnArgs", "TfdPanelMambaArgs",
        "TfdPanelGqaArgs")})
    test_abi.test_ctypes_structs_match_c_layout(tmp_path)


def _close(got, want, name):
    g, w = got.double(), want.double()
    off = float((g - w).norm() / w.norm().clamp(min=1e-30))
    assert off <= 2e-2, (name, off)


def _engine(model, rows, device, steps):
    if model == "qwen3_5":
        cfg = Q.Qwen35Config(layers=5, experts=8, top_k=8, vocab=512)
        return Q.Qwen35Engine(cfg, Q.synthetic_weights(cfg, 3, device), rows=rows, device=device,
                              max_steps=steps)
    cfg = G.GraniteConfig(layers=4, attention_layers=(1, 3), experts=8, top_k=8, vocab=512)
    return G.GraniteEngine(cfg, G.synthetic_weights(cfg, 3, device), rows=rows, device=device,
                           max_steps=steps)


def _left(eng):
    """What the next step reads."""
    out = {"pos": eng.pos.clone(), "ids": eng.ids.clone(), "emb": eng.emb.clone()}
    for i in eng.state:
        out[f"state {i}"] = eng.state[i].clone()
        out[f"window {i}"] = eng.conv[i][eng._cur].clone()
    for i in eng.kpool:
        out[f"k {i}"], out[f"v {i}"] = eng.kpool[i].clone(), eng.vpool[i].clone()
    return out


# no pass at all (one position is the walk's own step); two rows a sequence (fewer than
# a window); whole scan chunks and one more; passes cut in the middle, the last of two
# rows a sequence or of one (its window reaches back past the pass); expert tiles of 64
# rows and a rest
@pytest.mark.gpu
@pytest.mark.parametrize("model", ["qwen3_5", "granite"])
@pytest.mark.parametrize("rows,n,most", [(1, 2, 1024), (3, 3, 1024), (1, 18, 1024), (5, 40, 1024),
                                         (2, 99, 64), (3, 66, 1024), (2, 98, 64),
                                         (1, 66, 64)])
def test_pass_is_the_walk(gpu_device, monkeypatch, model, rows, n, most):
    monkeypatch.setattr(P, "MAX_PASS", most)
    eng = _engine(model, rows, gpu_device, n + 8)
    assert (P.Qwen35Pass if model == "qwen3_5" else P.GranitePass).takes(eng)
    g = torch.Generator().manual_seed(n)
    prompts = [torch.randint(0, 512, (n,), generator=g).tolist() for _ in range(rows)]
    eng._load_prompts(prompts)
    for pool in (*eng.kpool.values(), *eng.vpool.values()):
        pool.zero_()                        # the capture's own steps left rows behind
    for _ in range(n - 1):
        eng.replay()
    walked = _left(eng)
    eng.replay()
    logits = eng.logits.clone()
    for pool in (*eng.kpool.values(), *eng.vpool.values()):
        pool.zero_()
    eng.prefill(prompts)
    eng.check_errors()
    got = _left(eng)
    for name in ("pos", "ids", "emb"):
        assert torch.equal(got[name], walked[name]), name
    for name, want in walked.items():
        if name not in ("pos", "ids", "emb"):
            _close(got[name], want, name)
    eng.replay()
    eng.check_errors()
    _close(eng.logits, logits, "logits")


@pytest.mark.gpu
def test_odd_sizes_are_walked(gpu_device):
    """An engine outside the passes' sizes (row-major fp8 experts at 17 sequences) is
    brought to the same place by the decode step."""
    eng = _engine("granite", 17, gpu_device, 16)
    assert not P.GranitePass.takes(eng)
    prompts = [[1, 2 + b, 3] for b in range(17)]
    eng.prefill(prompts)
    assert eng.pos.tolist() == [2] * 17 and eng.ids.tolist() == [3] * 17


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["qwen3_5", "granite"])
def test_an_engine_that_prefilled_is_freed_when_dropped(gpu_device, model):
    """The engine and its pass hold no cycle: its device memory goes with the last
    reference, not with a later garbage collection."""
    import gc
    import weakref

    eng = _engine(model, 1, gpu_device, 12)
    gc.collect()
    gc.disable()
    try:
        eng.prefill([list(range(1, 9))])
        gone = weakref.ref(eng)
        del eng
        assert gone() is None
    finally:
        gc.enable()
