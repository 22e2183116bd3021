"""What a program that decodes with this framework has it do, as measurable cases.

Listed cases and the calls behind them:

* ``decode``: one Qwen3-1.7B-architecture sequence, token by token (``Engine``, the
  XCD-partitioned kernel), half the model's layers and its head;
* ``batch``: up to 32 sequences stepping together (``BatchEngine``), eight layers of
  the same model and its head;
* ``prompt`` / ``prompts``: the time to a first token -- prompts prefilled, then one
  decode step (``Engine`` and ``BatchEngine``), eight layers and the head;
* ``attention``: one layer's batched paged attention over long contexts;
* ``layer35`` / ``layerg``: one whole hybrid layer (Qwen3.5's gated DeltaNet + MoE,
  Granite's Mamba2 + fp8 MoE) as a program that binds the C ABI captures it: one
  graph of the entries the engines call;
* ``gqa``: one full-attention layer of the hybrids over long contexts;
* ``prompt35`` / ``promptg``: the hybrids' prompts (``prefill``, then one step), a
  four-layer cut with every kind of layer.

Everything a case reads is drawn from its seed on the GPU.  Recurrent steps feed
given tokens only (never the engine's own picks), so one rounding that settles a
near-tie another way does not change the rest of a run.
"""
from __future__ import annotations

import math

import torch

from tilefoundry_amd import _lib
from tilefoundry_amd._lib import lib, ptr
from tilefoundry_amd.hybrid import granite as G
from tilefoundry_amd.hybrid import qwen3_5 as Q
from tilefoundry_amd.qwen3 import QWEN3_1_7B
from tilefoundry_amd.qwen3.batch_engine import BatchEngine
from tilefoundry_amd.qwen3.engine import Engine, bf16_scale
from tilefoundry_amd.qwen3.prefill import attention_splits

BF, F32, F64, I32 = torch.bfloat16, torch.float32, torch.float64, torch.int32
DEV = "cuda:0"
HALF = 14          # layers of the batch-1 decode: 28 carry roundings past 3% of the logits
CUT = 8            # layers of the other Qwen3 cases
CUT_VOCAB = 24832  # a tenth of Qwen3.5's vocabulary, for its four-layer cut


# --------------------------------------------------------------------- the cases
def listed():
    return [
        # one user, one token at a time: 48 steps
        {"name": "decode b1", "kind": "decode", "tokens": 48},
        # a full batch over short chat contexts: projections, head, launches
        {"name": "decode b32", "kind": "batch", "rows": 32, "tokens": 24},
        # the attention of 32 sequences near 4,096 positions, each at its own depth
        {"name": "paged attention b32 4k", "kind": "attention", "rows": 32, "ctx": 4100},
        # a chat question: the first token after 91 prompt tokens
        {"name": "prompt 91", "kind": "prompt", "tokens": 91},
        # a document: the first token after 4,001 prompt tokens
        {"name": "prompt 4k", "kind": "prompt", "tokens": 4001},
        # eight users' prompts of different lengths arriving together
        {"name": "prompts b8 ragged", "kind": "prompts", "rows": 8, "tokens": 700},
        # one Qwen3.5 gated-DeltaNet layer at the workload's batch, and for one user
        {"name": "qwen3.5 layer b16", "kind": "layer35", "rows": 16},
        {"name": "qwen3.5 layer b1", "kind": "layer35", "rows": 1},
        # a Qwen3.5 prompt
        {"name": "qwen3.5 prompt 250", "kind": "prompt35", "rows": 1, "tokens": 250},
        # one Granite Mamba2 layer at the workload's batch
        {"name": "granite layer b8", "kind": "layerg", "rows": 8},
        # Granite's attention over 8,192-position contexts
        {"name": "granite attention b8 8k", "kind": "gqa", "model": "granite", "rows": 8,
         "ctx": 8190},
        # a Granite prompt
        {"name": "granite prompt 190", "kind": "promptg", "rows": 1, "tokens": 190},
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "batch", "attention", "prompt", "prompt", "prompts", "layer35",
                       "prompt35", "layerg", "gqa", "promptg"])
    if kind == "decode":
        return {"kind": kind, "tokens": _spread(rng, 9, 48)}
    if kind == "batch":
        return {"kind": kind, "rows": _spread(rng, 1, 32), "tokens": _spread(rng, 9, 24)}
    if kind == "attention":
        return {"kind": kind, "rows": _spread(rng, 2, 32), "ctx": _spread(rng, 100, 4100)}
    if kind == "prompt":
        return {"kind": kind, "tokens": _spread(rng, 17, 4000)}
    if kind == "prompts":
        return {"kind": kind, "rows": rng.randint(2, 8), "tokens": _spread(rng, 40, 700)}
    if kind == "layer35":
        return {"kind": kind, "rows": _spread(rng, 1, 32)}
    if kind == "layerg":
        return {"kind": kind, "rows": _spread(rng, 1, 32)}
    if kind == "gqa":
        model = rng.choice(["granite", "qwen3.5"])
        return {"kind": kind, "model": model, "rows": _spread(rng, 1, 16),
                "ctx": _spread(rng, 200, 8190 if model == "granite" else 2080)}
    rows = rng.choice([1, 1, 2, 3])
    return {"kind": kind, "rows": rows, "tokens": _spread(rng, 20, 250 // rows)}


# ------------------------------------------------------------------ drawn inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _rn(g, *shape, s=1.0, dtype=BF):
    return (torch.randn(*shape, generator=g, device=DEV) * s).to(dtype)


def _ids(seed, n, vocab):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


def _qwen3_weights(cfg, seed):
    """Random-init weights N(0, 0.02) with norm scales near 1, canonical names, the
    projections drawn (out, in) and handed over as (1, in, out) views, a tied head.
    Token rows are drawn near 1, so that the residual stream outweighs one layer's
    contribution as it does in a trained deep model (rows of 0.02 make every layer
    amplify the roundings of the one before)."""
    g = _gen(seed)
    h, i = cfg.hidden_size, cfg.intermediate_size
    w = {"w_embed": _rn(g, cfg.vocab_size, h)}
    w["w_head"] = w["w_embed"].t()
    shapes = {"w_q": (cfg.q_size, h), "w_k": (cfg.kv_size, h), "w_v": (cfg.kv_size, h),
              "w_o": (h, cfg.q_size), "w_gate": (i, h), "w_up": (i, h), "w_down": (h, i)}
    norms = {"gamma_in": h, "gamma_post": h, "gamma_q": cfg.head_dim, "gamma_k": cfg.head_dim}
    for layer in range(cfg.num_hidden_layers):
        for n, s in shapes.items():
            w[f"layer{layer}.{n}"] = _rn(g, *s, s=0.02).t().unsqueeze(0)
        for n, s in norms.items():
            w[f"layer{layer}.{n}"] = (1 + _rn(g, s, s=0.05, dtype=F32)).to(BF)
    w["gamma_final"] = (1 + _rn(g, h, s=0.05, dtype=F32)).to(BF)
    return w


def _qwen3(case):
    return QWEN3_1_7B.with_(num_hidden_layers=HALF if case["kind"] == "decode" else CUT)


def _prompts(case, seed, vocab):
    """Token ids per sequence: of one length, or spread below it for ``prompts``."""
    rows, n = case.get("rows", 1), case["tokens"]
    if case["kind"] != "prompts":
        return [_ids(seed * 1000 + b, n, vocab) for b in range(rows)]
    g = torch.Generator().manual_seed(seed)
    lens = torch.randint(max(8, n // 8), n + 1, (rows,), generator=g).tolist()
    return [_ids(seed * 1000 + b, m, vocab) for b, m in enumerate(lens)]


def _ragged(case, seed):
    """A position per sequence, from three quarters of the context to all of it."""
    g = torch.Generator().manual_seed(seed)
    return torch.randint(case["ctx"] * 3 // 4, case["ctx"], (case["rows"],), generator=g)


def _rope(theta, dim, rows, f64=False):
    dt = F64 if f64 else F32
    inv = 1.0 / theta ** (torch.arange(0, dim, 2, dtype=dt) / dim)
    ph = torch.outer(torch.arange(rows, dtype=dt), inv)
    ph = torch.cat((ph, ph), dim=-1)
    return ph.cos().to(BF).to(DEV), ph.sin().to(BF).to(DEV)


def _attention_inputs(case, seed):
    """One layer's q/k/v rows, norm scales and filled page pools at ragged depths."""
    g = _gen(seed)
    c = {"attention": (16, 8, 128), "granite": (32, 8, 128), "qwen3.5": (16, 2, 256)}
    HQ, HKV, D = c[case.get("model", case["kind"])]
    B = case["rows"]
    pages = -(-case["ctx"] // 64) * 4
    d = {"HQ": HQ, "HKV": HKV, "D": D, "pages": pages, "pos": _ragged(case, seed).to(I32).to(DEV)}
    d["table"] = torch.randperm(B * pages, generator=torch.Generator().manual_seed(seed)).view(
        B, pages).to(I32).to(DEV)
    d["k"], d["v"] = _rn(g, B * pages, HKV, 16, D), _rn(g, B * pages, HKV, 16, D, s=0.7)
    extra = 2 if case.get("model") == "qwen3.5" else 1        # Qwen3.5: an output gate per head
    d["qkv"] = _rn(g, B, (extra * HQ + 2 * HKV) * D)
    d["gq"] = (1 + _rn(g, D, s=0.05, dtype=F32)).to(BF)
    d["gk"] = (1 + _rn(g, D, s=0.05, dtype=F32)).to(BF)
    return d


def _layer_cfg(case):
    if case["kind"] == "layer35":
        return Q.Qwen35Config(layers=1, vocab=64)
    if case["kind"] == "layerg":
        return G.GraniteConfig(layers=1, attention_layers=(), vocab=64)
    if case["kind"] == "prompt35":
        return Q.Qwen35Config(layers=4, vocab=CUT_VOCAB)
    return G.GraniteConfig(layers=4, attention_layers=(1,), vocab=CUT_VOCAB)


def _hybrid_weights(case, seed):
    """The engines' synthetic weights, the token rows drawn so that the residual
    stream starts near 1 (as ``_qwen3_weights``; Granite multiplies its rows by 12)."""
    cfg = _layer_cfg(case)
    step35 = case["kind"].endswith("35")
    w = (Q if step35 else G).synthetic_weights(cfg, seed, DEV)
    w["embed"] = _rn(_gen(seed + 77), cfg.vocab, cfg.hidden, s=1.0 if step35 else 0.1)
    return cfg, w


def _layer_inputs(case, seed, cfg):
    """A token row per sequence and the mixer's state and window before the step."""
    g = _gen(seed + 5)
    B, x = case["rows"], {}
    if case["kind"] == "layer35":
        x["emb"] = _rn(g, B, cfg.hidden)
        x["state"] = _rn(g, B, cfg.lin_value_heads, cfg.lin_key_dim, cfg.lin_value_dim, s=0.1,
                         dtype=F32)
        x["conv"] = _rn(g, B, cfg.conv_dim, 3).float()
    else:
        x["emb"] = _rn(g, B, cfg.hidden, s=0.1)
        x["state"] = _rn(g, B, cfg.mamba_heads, cfg.mamba_head_dim, cfg.d_state, s=0.1, dtype=F32)
        x["conv"] = _rn(g, B, cfg.conv_dim, 3)
    return x


# ------------------------------------------------------------------------ prepare
def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "kind": kind}
    if kind in ("decode", "prompt"):
        cfg = _qwen3(case)
        s["prompt"] = _prompts(case, seed, cfg.vocab_size)[0]
        s["eng"] = Engine(cfg, _qwen3_weights(cfg, seed), device=DEV, max_new=8,
                          prompt_room=case["tokens"], mode="xcd")
        if kind == "prompt":
            s["eng"].prefill(s["prompt"][:2])         # lays the prefill's weights out
    elif kind in ("batch", "prompts"):
        cfg = _qwen3(case)
        s["prompts"] = _prompts(case, seed, cfg.vocab_size)
        s["eng"] = BatchEngine(cfg, _qwen3_weights(cfg, seed), batch=case["rows"], device=DEV,
                               max_new=8, prompt_room=case["tokens"])
        if kind == "prompts":
            s["eng"].prefill([p[:2] for p in s["prompts"]])
    elif kind in ("prompt35", "promptg"):
        cfg, w = _hybrid_weights(case, seed)
        cls = Q.Qwen35Engine if kind == "prompt35" else G.GraniteEngine
        s["eng"] = cls(cfg, w, rows=case["rows"], device=DEV, max_steps=case["tokens"] + 8)
        s["prompts"] = _prompts(case, seed, cfg.vocab)
        s["eng"].prefill([p[:2] for p in s["prompts"]])
    elif kind == "attention":
        _prepare_attention(case, seed, s)
    elif kind == "gqa":
        _prepare_gqa(case, seed, s)
    else:
        cfg, w = _hybrid_weights(case, seed)
        x = _layer_inputs(case, seed, cfg)
        before = x["state"].clone()
        layer = (_Layer35 if kind == "layer35" else _LayerGranite)(cfg, w, case["rows"], x)
        s["layer"], s["graph"] = layer, _captured(layer.launch)
        layer.state.copy_(before)                     # the run before the recording advanced it
    return s


def _captured(launch):
    """*launch* on the current stream, recorded into a graph after one plain run (as
    the engines capture their steps)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        launch()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch()
    return graph


def _z(*shape, dtype=F32):
    return torch.zeros(*shape, dtype=dtype, device=DEV)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _prepare_attention(case, seed, s):
    d, B = _attention_inputs(case, seed), case["rows"]
    cap = d["pages"] * 16
    nsplit = attention_splits(B, d["HKV"], cap)
    cos, sin = _rope(QWEN3_1_7B.rope_theta, d["D"], cap)
    d.update(cos=cos, sin=sin, cap=cap, nsplit=nsplit, B=B, scores=_z(B, d["HQ"], cap),
             smax=_z(B, nsplit, d["HQ"]), snew=_z(B, d["HQ"]), psum=_z(B, nsplit, d["HQ"]),
             pout=_z(B, nsplit, d["HQ"], d["D"]), counters=_z(B, d["HKV"], dtype=I32),
             out=_z(32 * d["HQ"] * d["D"], dtype=BF), err=_z(1, dtype=I32))
    s["d"] = d


def _run_attention(d):
    L, s = lib(), _stream()
    ldq, eps = d["qkv"].shape[1], QWEN3_1_7B.rms_norm_eps
    L.tfd_attn_rope_scores_paged_batched(
        ptr(d["qkv"]), ldq, ptr(d["gq"]), ptr(d["gk"]), ptr(d["cos"]), ptr(d["sin"]), d["cap"],
        ptr(d["pos"]), ptr(d["table"]), d["pages"], ptr(d["k"]), ptr(d["v"]), d["k"].shape[0],
        d["B"], d["HQ"], d["HKV"], d["D"], bf16_scale(d["D"]), eps, ptr(d["scores"]), d["cap"],
        ptr(d["smax"]), ptr(d["snew"]), d["nsplit"], 0, ptr(d["err"]), s)
    L.tfd_attn_pv_combine_paged_batched(
        ptr(d["qkv"]), ldq, ptr(d["pos"]), ptr(d["table"]), d["pages"], ptr(d["v"]),
        d["v"].shape[0], d["B"], d["HQ"], d["HKV"], d["D"], ptr(d["scores"]), d["cap"],
        ptr(d["smax"]), ptr(d["snew"]), ptr(d["psum"]), ptr(d["pout"]), d["nsplit"], 0,
        ptr(d["counters"]), ptr(d["out"]), ptr(d["err"]), s)
    return {"attn": d["out"], "k": d["k"], "v": d["v"]}


def _prepare_gqa(case, seed, s):
    d, B = _attention_inputs(case, seed), case["rows"]
    granite = case["model"] == "granite"
    cap = d["pages"] * 16
    if not granite:
        d["qkv"] = d["qkv"].float()
    nsplit = Q.attention_splits(B, d["HKV"], cap)
    d.update(out=_z(32 * d["HQ"] * d["D"], dtype=BF), err=_z(1, dtype=I32),
             scores=_z(B * d["HQ"] * cap), stats=_z(B * d["HQ"] * nsplit * 2),
             part=_z(B * d["HQ"] * nsplit * d["D"]), counters=_z(B * d["HKV"], dtype=I32))
    a = _lib.TfdGqaArgs()
    a.qkv, a.ldq = ptr(d["qkv"]), d["qkv"].shape[1]
    if not granite:
        d["cos"], d["sin"] = _rope(Q.Qwen35Config.rope_theta, Q.Qwen35Config.rot_dim, cap, True)
        a.gamma_q, a.gamma_k = ptr(d["gq"]), ptr(d["gk"])
        a.cos_table, a.sin_table = ptr(d["cos"]), ptr(d["sin"])
        a.rope_rows, a.rot_dim = cap, Q.Qwen35Config.rot_dim
    a.pos, a.page_table, a.max_pages = ptr(d["pos"]), ptr(d["table"]), d["pages"]
    a.k_pool, a.v_pool, a.num_pages = ptr(d["k"]), ptr(d["v"]), d["k"].shape[0]
    a.rows, a.heads, a.kv_heads, a.head_dim = B, d["HQ"], d["HKV"], d["D"]
    a.scale = G.GraniteConfig.attention_multiplier if granite else d["D"] ** -0.5
    a.eps = G.GraniteConfig.eps if granite else Q.Qwen35Config.eps
    a.scores, a.score_stride, a.stats, a.part = ptr(d["scores"]), cap, ptr(d["stats"]), \
        ptr(d["part"])
    a.counters, a.nsplit, a.split_len = ptr(d["counters"]), nsplit, 0
    a.out, a.err = ptr(d["out"]), ptr(d["err"])
    a.policy = _lib.POLICY_BF16 if granite else _lib.POLICY_F32
    s["d"], s["args"] = d, a


class _Layer35:
    """One Qwen3.5 gated-DeltaNet layer at one token per sequence: the entries the
    engine calls, in its two forms (up to 4 rows; more)."""

    def __init__(self, cfg, w, rows, x):
        self.cfg, self.B = cfg, rows
        self.w = {k[len("layer0."):]: v for k, v in w.items() if k.startswith("layer0.")}
        self.small = rows <= _lib.SMALL_ROWS
        self.emb, self.state, self.conv_in = x["emb"], x["state"], x["conv"]
        self.conv_out = torch.zeros_like(self.conv_in)
        if not self.small:
            for n in ("w_in", "w_out", "w_router"):
                N, K = self.w[n].shape
                packed = torch.empty(-(-N // 16) * 16 * K, dtype=BF, device=DEV)
                lib().tfd_pack_skinny_bf16(ptr(self.w[n]), K, N, K, ptr(packed), _stream())
                self.w[n] = packed
        c, B, H, k = cfg, rows, cfg.hidden, cfg.top_k
        self.hidden, self.xn, self.xm = _z(B, H), _z(32 * H, dtype=BF), _z(B, H, dtype=BF)
        self.proj, self.mix = _z(B, c.gdn_in), _z(32 * c.value_dim, dtype=BF)
        self.read, self.rlog = _z(B, c.value_dim), _z(B, c.experts)
        self.work = _z(1 << 21)
        g = self.g = _lib.TfdGdnArgs()
        g.proj, g.proj_ld, g.conv_in, g.conv_out = ptr(self.proj), c.gdn_in, ptr(self.conv_in), \
            ptr(self.conv_out)
        g.state, g.conv_w, g.a_log = ptr(self.state), ptr(self.w["conv_w"]), ptr(self.w["a_log"])
        g.dt_bias, g.gamma, g.out = ptr(self.w["dt_bias"]), ptr(self.w["gamma_gdn"]), ptr(self.mix)
        g.rows, g.key_heads, g.value_heads = B, c.lin_key_heads, c.lin_value_heads
        g.head_k_dim, g.head_v_dim, g.conv_kernel = c.lin_key_dim, c.lin_value_dim, c.conv_kernel
        g.l2_eps, g.rms_eps = 1e-6, c.eps
        self.m = _moe_args(self, c, k, _lib.MOE_ROUTE_SOFTMAX_TOPK)
        self.m.out, self.m.accumulate = ptr(self.hidden), 1
        self.m.w_shared_scale = ptr(self.w["w_shared_scale"])
        self.m.fp8, self.m.policy = 0, _lib.POLICY_F32

    def _rows_gemv(self, kind, x, ldx, w, K, N, out, ldo, gamma, resid=False, x_rows=None):
        a = _lib.TfdRowGemvArgs()
        a.x, a.ldx, a.x_kind, a.gamma, a.head_dim = ptr(x), ldx, kind, ptr(gamma), \
            self.cfg.lin_value_dim
        a.eps, a.w, a.K, a.N, a.out, a.ldo = self.cfg.eps, ptr(w), K, N, ptr(out), ldo
        if kind == _lib.ROWX_GATED_F32:
            a.gate, a.ldg = ptr(self.proj) + 4 * self.cfg.conv_dim, self.cfg.gdn_in
        a.epilogue = _lib.EPI_RESID_F32 if resid else _lib.EPI_LOGITS
        if x_rows is not None:
            a.x_rows, a.ldxr = ptr(x_rows), K
        a.rows = self.B
        lib().tfd_rowgemv_bf16(Q.ctypes_addr(a), _stream())

    def _gemm(self, x, w, K, N, out, ldo, resid=None):
        lib().tfd_gemm_skinny_bf16(
            ptr(x), ptr(w), self.B, K, N, _lib.EPI_LOGITS if resid is None else
            _lib.EPI_RESID_F32, None if resid is None else ptr(resid),
            0 if resid is None else ldo, ptr(out), ldo, ptr(self.work), self.work.numel(),
            _stream())

    def launch(self):
        L, s, c, w, B, H = lib(), _stream(), self.cfg, self.w, self.B, self.cfg.hidden
        L.tfd_bf16_to_f32_rows(ptr(self.emb), H, ptr(self.hidden), H, B, H, s)
        if self.small:
            self._rows_gemv(_lib.ROWX_NORM_F32, self.hidden, H, w["w_in"], H, c.gdn_in,
                            self.proj, c.gdn_in, w["gamma_in"])
            L.tfd_gdn_step_cols(Q.ctypes_addr(self.g), ptr(self.read), c.value_dim, s)
            self._rows_gemv(_lib.ROWX_GATED_F32, self.read, c.value_dim, w["w_out"], c.value_dim,
                            H, self.hidden, H, w["gamma_gdn"], resid=True)
            self._rows_gemv(_lib.ROWX_NORM_F32, self.hidden, H, w["w_router"], H, c.experts,
                            self.rlog, c.experts, w["gamma_post"], x_rows=self.xm)
            L.tfd_moe_experts_small(Q.ctypes_addr(self.m), s)
            return
        L.tfd_rmsnorm_f32_rows(ptr(self.hidden), H, ptr(w["gamma_in"]), None, 0, ptr(self.xn), B,
                               H, c.eps, s)
        self._gemm(self.xn, w["w_in"], H, c.gdn_in, self.proj, c.gdn_in)
        L.tfd_gdn_step(Q.ctypes_addr(self.g), s)
        self._gemm(self.mix, w["w_out"], c.value_dim, H, self.hidden, H, resid=self.hidden)
        L.tfd_rmsnorm_f32_rows(ptr(self.hidden), H, ptr(w["gamma_post"]), ptr(self.xm), H,
                               ptr(self.xn), B, H, c.eps, s)
        self._gemm(self.xn, w["w_router"], H, c.experts, self.rlog, c.experts)
        L.tfd_moe_experts(Q.ctypes_addr(self.m), s)


def _moe_args(layer, c, k, route):
    """TfdMoeArgs of a layer's own buffers (kept on the layer)."""
    B, w, a = layer.B, layer.w, _lib.TfdMoeArgs()
    ld = max(c.moe_inter, c.shared_inter)
    layer.rw, layer.ridx = _z(B, k), _z(B, k, dtype=I32)
    layer.moe_hidden, layer.moe_scale = _z(B, k + 1, ld, dtype=BF), _z(B)
    layer.moe_partial = _z(B, k + 1, c.hidden)
    layer.groups = _z(_lib.moe_group_words(c.experts, B), dtype=I32)
    layer.err = _z(1, dtype=I32)
    a.x, a.weights, a.idx = ptr(layer.xm), ptr(layer.rw), ptr(layer.ridx)
    a.w_gate, a.w_up, a.w_down = ptr(w["w_gate"]), ptr(w["w_up"]), ptr(w["w_down"])
    a.w_shared_in, a.w_shared_out = ptr(w["w_shared_in"]), ptr(w["w_shared_out"])
    a.hidden, a.shared_scale = ptr(layer.moe_hidden), ptr(layer.moe_scale)
    a.partial, a.groups, a.err = ptr(layer.moe_partial), ptr(layer.groups), ptr(layer.err)
    a.rows, a.k, a.experts, a.hidden_size = B, k, c.experts, c.hidden
    a.inter, a.shared_inter, a.hidden_ld = c.moe_inter, c.shared_inter, ld
    a.logits, a.ldl, a.route = ptr(layer.rlog), c.experts, route
    return a


class _LayerGranite:
    """One Granite Mamba2 layer at one token per sequence, fp8 weights: the entries
    the engine calls (packed experts up to 16 rows, the router with its norm up to 8)."""

    def __init__(self, cfg, w, rows, x):
        self.cfg, self.B = c, B = cfg, rows
        self.w = {k[len("layer0."):]: v for k, v in w.items() if k.startswith("layer0.")}
        self.emb, self.state, self.conv_in = x["emb"], x["state"], x["conv"]
        self.conv_out = torch.zeros_like(self.conv_in)
        self.packed = _lib.moe_packed_fits(B, c.top_k, c.hidden, c.moe_inter, c.shared_inter)
        names = ["w_in", "w_out", "w_router"]
        if self.packed:
            names += ["w_gate", "w_up", "w_down", "w_shared_in", "w_shared_out"]
        for n in names:
            N, K = self.w[n].shape
            out = torch.empty(-(-N // 16) * 16 * K, dtype=torch.uint8, device=DEV)
            lib().tfd_pack_skinny_fp8(ptr(self.w[n]), K, N, K, ptr(out), _stream())
            self.w[n] = out
        H = c.hidden
        self.hidden, self.xn, self.xm = _z(B, H, dtype=BF), _z(32 * H, dtype=BF), \
            _z(B, H, dtype=BF)
        self.proj, self.mix = _z(B, c.mamba_in, dtype=BF), _z(32 * c.d_inner, dtype=BF)
        self.rlog, self.gated, self.ssq = _z(B, c.experts), _z(B, c.d_inner), _z(B, c.mamba_heads)
        a = self.a = _lib.TfdMambaArgs()
        a.proj, a.proj_ld, a.conv_in, a.conv_out = ptr(self.proj), c.mamba_in, \
            ptr(self.conv_in), ptr(self.conv_out)
        a.state, a.conv_w, a.conv_b = ptr(self.state), ptr(self.w["conv_w"]), ptr(self.w["conv_b"])
        a.a_log, a.dt_bias, a.d_skip = ptr(self.w["a_log"]), ptr(self.w["dt_bias"]), \
            ptr(self.w["d_skip"])
        a.gamma, a.gated, a.ssq, a.out = ptr(self.w["gamma_ssm"]), ptr(self.gated), \
            ptr(self.ssq), ptr(self.mix)
        a.rows, a.heads, a.head_dim, a.state_dim = B, c.mamba_heads, c.mamba_head_dim, c.d_state
        a.groups, a.conv_kernel, a.eps = 1, c.conv_kernel, c.eps
        m = self.m = _moe_args(self, c, c.top_k, _lib.MOE_ROUTE_TOPK_SOFTMAX)
        m.s_gate, m.s_up, m.s_down = (ptr(self.w[n]) for n in ("s_gate", "s_up", "s_down"))
        m.s_shared_in, m.s_shared_out = ptr(self.w["w_shared_in_scale"]), \
            ptr(self.w["w_shared_out_scale"])
        m.fp8, m.policy = 1, _lib.POLICY_BF16
        m.resid, m.resid_mult = ptr(self.hidden), c.residual_multiplier
        p = self.p = _lib.TfdProj8NormArgs()
        p.x, p.ldx, p.gamma, p.eps = ptr(self.hidden), H, ptr(self.w["gamma_post"]), c.eps
        p.x_rows, p.ldxr, p.w, p.scale = ptr(self.xm), H, ptr(self.w["w_router"]), \
            ptr(self.w["w_router_scale"])
        p.rows, p.K, p.N = B, H, c.experts
        p.out, p.ldo, p.epilogue = ptr(self.rlog), c.experts, _lib.EPI_LOGITS

    def launch(self):
        L, s, c, w, B, H = lib(), _stream(), self.cfg, self.w, self.B, self.cfg.hidden
        L.tfd_scaled_add_rows(None, 0, ptr(self.emb), H, 0, c.embedding_multiplier,
                              ptr(self.hidden), H, B, H, s)
        L.tfd_tf_rmsnorm_rows_bf16(ptr(self.hidden), H, ptr(w["gamma_in"]), None, 0, ptr(self.xn),
                                   B, H, c.eps, s)
        L.tfd_gemm_skinny_fp8(ptr(self.xn), ptr(w["w_in"]), ptr(w["w_in_scale"]), B, H,
                              c.mamba_in, _lib.EPI_STORE, None, 0, ptr(self.proj), c.mamba_in, s)
        L.tfd_mamba_step(Q.ctypes_addr(self.a), s)
        L.tfd_gemm_skinny_fp8_resid_scaled(
            ptr(self.mix), ptr(w["w_out"]), ptr(w["w_out_scale"]), B, c.d_inner, H,
            ptr(self.hidden), H, c.residual_multiplier, ptr(self.hidden), H, s)
        if B <= _lib.PROJ8_ROWS:
            L.tfd_proj8_norm(Q.ctypes_addr(self.p), s)
        else:
            L.tfd_tf_rmsnorm_rows_bf16(ptr(self.hidden), H, ptr(w["gamma_post"]), ptr(self.xm), H,
                                       ptr(self.xn), B, H, c.eps, s)
            L.tfd_gemm_skinny_fp8(ptr(self.xn), ptr(w["w_router"]), ptr(w["w_router_scale"]), B,
                                  H, c.experts, _lib.EPI_LOGITS, None, 0, ptr(self.rlog),
                                  c.experts, s)
        if self.packed:
            L.tfd_moe_experts_packed(Q.ctypes_addr(self.m), s)
        else:
            L.tfd_moe_experts(Q.ctypes_addr(self.m), s)


# ---------------------------------------------------------------------------- run
def run(s):
    kind, eng = s["kind"], s.get("eng")
    if kind == "decode":
        return {"logits": eng.logits_for(s["prompt"]), "k": eng.kpool, "v": eng.vpool}
    if kind == "prompt":
        eng.generate(s["prompt"], 1, prefill=True)
        return {"logits": eng.logits, "k": eng.kpool, "v": eng.vpool}
    if kind in ("batch", "prompts"):
        eng.generate(s["prompts"], 1, prefill=kind == "prompts")
        return {"logits": eng.logits, "k": eng.kpool, "v": eng.vpool}
    if kind in ("prompt35", "promptg"):
        eng.prefill(s["prompts"])
        eng.replay()
        return {"logits": eng.logits, "k": eng.kpool, "v": eng.vpool, "state": eng.state}
    if kind == "attention":
        return _run_attention(s["d"])
    if kind == "gqa":
        lib().tfd_gqa_decode(Q.ctypes_addr(s["args"]), _stream())
        return {"attn": s["d"]["out"], "k": s["d"]["k"], "v": s["d"]["v"]}
    s["graph"].replay()
    layer = s["layer"]
    return {"hidden": layer.hidden, "state": layer.state, "window": layer.conv_out}


# --------------------------------------------------------------------------- work
def work(case):
    """Weights read once per step that decodes (once per prompt that is prefilled),
    cache and state read and written once, every product of the model."""
    kind, B = case["kind"], case.get("rows", 1)
    if kind in ("decode", "batch", "prompt", "prompts"):
        cfg = _qwen3(case)
        n = case["tokens"]
        total = B * n if kind != "prompts" else int(B * n * 0.56)      # mean drawn length
        layer = cfg.layer_params() * cfg.num_hidden_layers
        head = cfg.vocab_size * cfg.hidden_size
        per = total / B
        kv = cfg.kv_bytes_per_position()
        attn = 4 * cfg.q_size * cfg.num_hidden_layers * B * per * per / 2
        if kind in ("decode", "batch"):                # a step per token
            return {"bytes": 2.0 * n * (layer + head) + B * kv * n * (n + 1) / 2,
                    "flops": 2.0 * total * (layer + head) + attn}
        return {"bytes": 2.0 * (layer + head) + kv * total * 2,
                "flops": 2.0 * total * layer + 2.0 * B * head + attn}
    if kind in ("attention", "gqa"):
        HQ, HKV, D = {"attention": (16, 8, 128), "granite": (32, 8, 128),
                      "qwen3.5": (16, 2, 256)}[case.get("model", kind)]
        positions = B * case["ctx"] * 7 / 8
        return {"bytes": 4.0 * HKV * D * positions + 4.0 * B * HQ * D,
                "flops": 4.0 * HQ * D * positions}
    cfg = _layer_cfg(case)
    T = case.get("tokens", 1)
    picked = min(1.0, 1 - (1 - cfg.top_k / cfg.experts) ** (B * T))   # share of experts read
    H = cfg.hidden
    expert, shared = 3 * cfg.moe_inter * H, 3 * cfg.shared_inter * H
    if kind.endswith("35"):
        size, mixers = 2, 3 if cfg.layers == 4 else 1
        mixer = cfg.gdn_in * H + H * cfg.value_dim
        attn = (cfg.attn_in * H + H * cfg.heads * cfg.head_dim) * (cfg.layers - mixers)
        state = mixers * B * 4 * cfg.lin_value_heads * cfg.lin_key_dim * cfg.lin_value_dim
        scan = mixers * 6 * cfg.lin_value_heads * cfg.lin_key_dim * cfg.lin_value_dim
    else:
        size, mixers = 1, 3 if cfg.layers == 4 else 1
        mixer = cfg.mamba_in * H + H * cfg.d_inner
        attn = (cfg.attn_in * H + H * cfg.heads * cfg.head_dim) * (cfg.layers - mixers)
        state = mixers * B * 4 * cfg.d_inner * cfg.d_state
        scan = mixers * 6 * cfg.d_inner * cfg.d_state
    head = 0 if T == 1 else cfg.vocab * H
    dense = mixers * mixer + attn + cfg.layers * (shared + cfg.experts * H)
    moe = cfg.layers * cfg.experts * expert * picked
    return {"bytes": size * (dense + moe) + 2.0 * head + 2 * state,
            "flops": 2.0 * B * (T * (dense + cfg.layers * cfg.top_k * expert) + head) +
            B * T * scan}


# ---------------------------------------------------------------------- tolerance
def tolerance(case):
    """bf16 outputs of f32 sums.  Stacked layers carry one layer's changed roundings
    through all that follow: the framework's own paths of different summation orders
    (batch-1 kernels, walked and prefilled prompts, row GEMVs and matrix-core GEMMs)
    differ by 0.9-1.6% in eight Qwen3 layers' logits and caches, by 0.5-1.9% in four
    hybrid layers'.  Single layers differ by the rounding of each product's inputs."""
    return {"attention": {"rel": 1.5e-2}, "gqa": {"rel": 1e-2}, "layer35": {"rel": 1e-2},
            "layerg": {"rel": 1e-2}}.get(case["kind"], {"rel": 3e-2})


# -------------------------------------------------------------- the values in f64
def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "batch", "prompt", "prompts"):
        return _exact_qwen3(case, seed)
    if kind in ("attention", "gqa"):
        return _exact_attention(case, seed)
    cfg, w = _hybrid_weights(case, seed)
    step35 = kind.endswith("35")
    if kind.startswith("layer"):
        x = _layer_inputs(case, seed, cfg)
        emb = x["emb"].double()[:, None]
        h, out = _exact_hybrid(cfg, w, emb if step35 else emb * cfg.embedding_multiplier, step35,
                               x["state"].double(), x["conv"].double())
        return {"hidden": h[:, 0], "state": out["state"][0], "window": out["window"][0]}
    prompts = torch.tensor(_prompts(case, seed, cfg.vocab), device=DEV)
    emb = w["embed"][prompts].double()
    h, out = _exact_hybrid(cfg, w, emb if step35 else emb * cfg.embedding_multiplier, step35)
    last = _rms(h[:, -1], w["gamma_final"], cfg.eps)
    head = w["head"] if step35 else w["embed"]
    logits = last @ head.double().t() / (1.0 if step35 else cfg.logits_scaling)
    pages = -(-(case["tokens"] + 8) // 16)
    table = torch.randperm(case["rows"] * pages, generator=torch.Generator().manual_seed(0)).view(
        case["rows"], pages).to(DEV)
    pools = {n: {i: _paged(c, table) for i, c in out[n].items()} for n in ("k", "v")}
    return {"logits": logits, "k": pools["k"], "v": pools["v"], "state": out["state"]}


def _rms(x, gamma, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * gamma.double()


def _paged(cache, table):
    """[B][P][HKV][D] caches as the pages [pages][HKV][16][D] that *table* places."""
    B, P, HKV, D = cache.shape
    pool = torch.zeros(table.numel(), HKV, 16, D, dtype=F64, device=DEV)
    p = torch.arange(P, device=DEV)
    for b in range(B):
        pool[table[b].long()[p // 16], :, p % 16] = cache[b]
    return pool


def _rotate(x, cos, sin):
    """Rotate-half RoPE of the first cos.shape[-1] dims; x [..., P, heads, D]."""
    rot = cos.shape[-1]
    r = x[..., :rot]
    half = torch.cat((-r[..., rot // 2:], r[..., :rot // 2]), -1)
    return torch.cat((r * cos[:, None] + half * sin[:, None], x[..., rot:]), -1)


def _causal(q, k, v, scale):
    """Causal attention of one sequence: q [P][HQ][D], k / v [P][HKV][D]."""
    P, HQ, D = q.shape
    rep = HQ // k.shape[1]
    out = torch.empty_like(q)
    late = torch.ones(P, P, dtype=torch.bool, device=DEV).triu(1)
    for h in range(HQ):
        s = (q[:, h] @ k[:, h // rep].t()) * scale
        out[:, h] = torch.softmax(s.masked_fill_(late, -math.inf), -1) @ v[:, h // rep]
    return out


def _exact_qwen3(case, seed):
    cfg = _qwen3(case)
    w, prompts = _qwen3_weights(cfg, seed), _prompts(case, seed, cfg.vocab_size)
    cap = -(-(case["tokens"] + 8) // 64) * 64
    B, D, pages = len(prompts), cfg.head_dim, cap // 16
    table = torch.randperm(B * pages, generator=torch.Generator().manual_seed(0)).view(B, pages)
    table = table.to(DEV)
    cos, sin = (t.double() for t in _rope(cfg.rope_theta, D, cap))
    xs = [w["w_embed"][torch.tensor(p, device=DEV)].double() for p in prompts]
    ks, vs, eps = [], [], cfg.rms_norm_eps
    for i in range(cfg.num_hidden_layers):
        m = {n: w[f"layer{i}.{n}"].double() for n in
             ("w_q", "w_k", "w_v", "w_o", "w_gate", "w_up", "w_down")}
        m = {n: t[0] for n, t in m.items()}
        gam = {n: w[f"layer{i}.{n}"] for n in ("gamma_in", "gamma_post", "gamma_q", "gamma_k")}
        kp = torch.zeros(B * pages, cfg.num_key_value_heads, 16, D, dtype=F64, device=DEV)
        vp = torch.zeros_like(kp)
        for b, x in enumerate(xs):
            P = x.shape[0]
            n = _rms(x, gam["gamma_in"], eps)
            q = _rms((n @ m["w_q"]).view(P, -1, D), gam["gamma_q"], eps)
            k = _rms((n @ m["w_k"]).view(P, -1, D), gam["gamma_k"], eps)
            v = (n @ m["w_v"]).view(P, -1, D)
            q, k = _rotate(q, cos[:P], sin[:P]), _rotate(k, cos[:P], sin[:P])
            at = torch.arange(P, device=DEV)
            kp[table[b].long()[at // 16], :, at % 16] = k
            vp[table[b].long()[at // 16], :, at % 16] = v
            x = x + _causal(q, k, v, bf16_scale(D)).reshape(P, -1) @ m["w_o"]
            n = _rms(x, gam["gamma_post"], eps)
            xs[b] = x + (torch.nn.functional.silu(n @ m["w_gate"]) * (n @ m["w_up"])) @ m["w_down"]
        ks.append(kp)
        vs.append(vp)
    last = _rms(torch.stack([x[-1] for x in xs]), w["gamma_final"], eps)
    logits = last @ w["w_embed"].double().t()
    if case["kind"] in ("decode", "prompt"):
        logits = logits[0]
    return {"logits": logits, "k": torch.stack(ks), "v": torch.stack(vs)}


def _exact_attention(case, seed):
    d, B = _attention_inputs(case, seed), case["rows"]
    HQ, HKV, D, model = d["HQ"], d["HKV"], d["D"], case.get("model", "qwen3")
    qkv, pos, cap = d["qkv"].double(), d["pos"].tolist(), d["pages"] * 16
    k_pool, v_pool = d["k"].double(), d["v"].double()
    out, scale, gate = [], bf16_scale(D), None
    if model == "qwen3":
        cos, sin = (t.double() for t in _rope(QWEN3_1_7B.rope_theta, D, cap))
    elif model == "qwen3.5":
        cos, sin = (t.double() for t in _rope(Q.Qwen35Config.rope_theta, Q.Qwen35Config.rot_dim,
                                              cap, True))
        scale = D ** -0.5
    else:
        scale = G.GraniteConfig.attention_multiplier
    nq = qkv.shape[1] // D - 2 * HKV
    for b in range(B):
        heads = qkv[b].view(-1, D)
        q, k, v = heads[:nq], heads[nq:nq + HKV], heads[nq + HKV:]
        if model == "qwen3.5":
            q, gate = q.reshape(HQ, 2, D).unbind(1)
        if model != "granite":
            at = slice(pos[b], pos[b] + 1)
            q, k = (_rotate(_rms(t, gm, 1e-6)[None], cos[at], sin[at])[0]
                    for t, gm in ((q, d["gq"]), (k, d["gk"])))
        p = torch.arange(pos[b], device=DEV)
        page = d["table"][b].long()
        past_k, past_v = (t[page[p // 16], :, p % 16] for t in (k_pool, v_pool))
        ks, vs = torch.cat((past_k, k[None])), torch.cat((past_v, v[None]))
        rep = HQ // HKV
        sc = torch.einsum("hd,phd->hp", q, ks.repeat_interleave(rep, 1)) * scale
        o = torch.einsum("hp,phd->hd", torch.softmax(sc, -1), vs.repeat_interleave(rep, 1))
        out.append((o * torch.sigmoid(gate) if gate is not None else o).reshape(-1))
        k_pool[page[pos[b] // 16], :, pos[b] % 16] = k
        v_pool[page[pos[b] // 16], :, pos[b] % 16] = v
    rows = torch.zeros(32, HQ * D, dtype=F64, device=DEV)
    rows[:B] = torch.stack(out)
    # operand order: block (2 s + h) holds rows 16 h + l % 16, columns 32 s + 8 (l / 16) ..
    blocks = rows.view(2, 16, HQ * D // 32, 4, 8).permute(2, 0, 3, 1, 4)
    return {"attn": blocks.reshape(-1), "k": k_pool, "v": v_pool}


def _experts(cfg, w, x, weights, idx, step35):
    """Routed + shared experts over tokens x [N][H]."""
    silu = torch.nn.functional.silu

    def mat(name, scale=None, e=None):
        t = w[name] if e is None else w[name].view(cfg.experts, -1, w[name].shape[-1])[e]
        if step35:
            return t.double()
        sc = w[scale] if e is None else w[scale].view(cfg.experts, -1)[e]
        return t.view(torch.float8_e4m3fn).double() * sc.double()[:, None]

    out = torch.zeros_like(x)
    for e in idx.unique().tolist():
        at = (idx == e).nonzero()
        t = x[at[:, 0]]
        h = silu(t @ mat("w_gate", "s_gate", e).t()) * (t @ mat("w_up", "s_up", e).t())
        out.index_add_(0, at[:, 0], (h @ mat("w_down", "s_down", e).t()) *
                       weights[at[:, 0], at[:, 1], None])
    both = x @ mat("w_shared_in", "w_shared_in_scale").t()
    g, u = both.chunk(2, -1)
    shared = (silu(g) * u) @ mat("w_shared_out", "w_shared_out_scale").t()
    if step35:
        shared = shared * torch.sigmoid(x @ w["w_shared_scale"].double())[:, None]
    return out + shared


def _exact_hybrid(cfg, weights, x, step35, state=None, window=None):
    """The layers over x [B][T][H] -> (x, caches, states and windows after them)."""
    B, T, H = x.shape
    out = {"k": {}, "v": {}, "state": {}, "window": {}}
    for i in range(cfg.layers):
        w = {k[len(f"layer{i}."):]: v for k, v in weights.items() if k.startswith(f"layer{i}.")}

        def lin(name, t):
            m = w[name].double() if step35 else \
                w[name].view(torch.float8_e4m3fn).double() * w[name + "_scale"].double()[:, None]
            return t @ m.t()

        proj = lin("w_in", _rms(x, w["gamma_in"], cfg.eps))
        if cfg.is_full(i) if step35 else cfg.is_attention(i):
            y = _exact_attend(cfg, w, proj, step35, out, i)
        else:
            mixer = _exact_gdn if step35 else _exact_mamba
            y, out["state"][i], out["window"][i] = mixer(cfg, w, proj, state, window)
        mult = 1.0 if step35 else cfg.residual_multiplier
        x = x + lin("w_out", y) * mult
        t = _rms(x, w["gamma_post"], cfg.eps).reshape(B * T, H)
        logits = lin("w_router", t)
        if step35:
            p, idx = torch.softmax(logits, -1).topk(cfg.top_k, -1)
            p = p / p.sum(-1, keepdim=True)
        else:
            p, idx = logits.topk(cfg.top_k, -1)
            p = torch.softmax(p, -1)
        x = x + _experts(cfg, w, t, p, idx, step35).view(B, T, H) * mult
    return x, out


def _exact_attend(cfg, w, proj, step35, out, i):
    B, T, _ = proj.shape
    HQ, HKV, D = cfg.heads, cfg.kv_heads, cfg.head_dim
    nq = HQ * (2 if step35 else 1)
    heads = proj.view(B, T, -1, D)[:, :, :nq + 2 * HKV]
    q, k, v = heads[:, :, :nq], heads[:, :, nq:nq + HKV], heads[:, :, nq + HKV:]
    gate, scale = 1.0, getattr(cfg, "attention_multiplier", D ** -0.5)
    if step35:
        q, gate = q.reshape(B, T, HQ, 2, D).unbind(3)
        gate = torch.sigmoid(gate).reshape(B, T, -1)
        cos, sin = (t.double() for t in _rope(cfg.rope_theta, cfg.rot_dim, T, True))
        q = _rotate(_rms(q, w["gamma_q"], cfg.eps), cos, sin)
        k = _rotate(_rms(k, w["gamma_k"], cfg.eps), cos, sin)
    out["k"][i], out["v"][i] = k, v
    return torch.stack([_causal(q[b], k[b], v[b], scale) for b in range(B)]).reshape(
        B, T, -1) * gate


def _conv(entry, window, w):
    """The depthwise causal convolution -> (values [B][T][C], the window after it)."""
    B, T, C = entry.shape
    past = torch.zeros(B, 3, C, dtype=F64, device=DEV) if window is None else window.transpose(1, 2)
    e = torch.cat((past, entry), 1)
    y = sum(e[:, j:j + T] * w.double()[:, j] for j in range(4))
    return y, e[:, -3:].transpose(1, 2)


def _exact_gdn(cfg, w, proj, state, window):
    B, T, _ = proj.shape
    hk, hv, d = cfg.lin_key_heads, cfg.lin_value_heads, cfg.lin_key_dim
    silu = torch.nn.functional.silu
    mixed, window = _conv(proj[..., :cfg.conv_dim], window, w["conv_w"])
    mixed = silu(mixed)
    z, b_raw, a_raw = proj[..., cfg.conv_dim:].split([cfg.value_dim, hv, hv], -1)
    q, k, v = mixed.split([cfg.key_dim, cfg.key_dim, cfg.value_dim], -1)
    q, k = (t.reshape(B, T, hk, d).repeat_interleave(hv // hk, 2) for t in (q, k))
    q, k = (t * torch.rsqrt(t.pow(2).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
    v, beta = v.reshape(B, T, hv, -1), torch.sigmoid(b_raw)
    g = -torch.exp(w["a_log"].double()) * torch.nn.functional.softplus(a_raw +
                                                                      w["dt_bias"].double())
    S = torch.zeros(B, hv, d, v.shape[-1], dtype=F64, device=DEV) if state is None else state
    read = []
    for t in range(T):
        S = S * torch.exp(g[:, t])[..., None, None]
        recalled = (S * k[:, t, :, :, None]).sum(2)
        S = S + k[:, t, :, :, None] * ((v[:, t] - recalled) * beta[:, t, :, None])[:, :, None]
        read.append((S * (q[:, t] * d ** -0.5)[..., None]).sum(2))
    r = _rms(torch.stack(read, 1), w["gamma_gdn"], cfg.eps)
    return (r * silu(z.reshape(r.shape))).reshape(B, T, -1), S, window


def _exact_mamba(cfg, w, proj, state, window):
    B, T, _ = proj.shape
    nh, pd, ns = cfg.mamba_heads, cfg.mamba_head_dim, cfg.d_state
    silu = torch.nn.functional.silu
    gate, entry, dt = proj.split([cfg.d_inner, cfg.conv_dim, nh], -1)
    mixed, window = _conv(entry, window, w["conv_w"])
    mixed = silu(mixed + w["conv_b"].double())
    x, bv, cv = mixed.split([cfg.d_inner, ns, ns], -1)
    x = x.reshape(B, T, nh, pd)
    dt = torch.nn.functional.softplus(dt + w["dt_bias"].double())
    decay = torch.exp(dt * -torch.exp(w["a_log"].double()))
    S = torch.zeros(B, nh, pd, ns, dtype=F64, device=DEV) if state is None else state
    ys = []
    for t in range(T):
        S = S * decay[:, t, :, None, None] + (dt[:, t, :, None] * x[:, t])[..., None] * \
            bv[:, t, None, None]
        ys.append((S * cv[:, t, None, None]).sum(-1) + x[:, t] * w["d_skip"].double()[:, None])
    y = torch.stack(ys, 1).reshape(B, T, -1) * silu(gate)
    return _rms(y, w["gamma_ssm"], cfg.eps), S, window
