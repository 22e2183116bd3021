"""Prompt passes of the hybrid engines: many positions through a layer at once.

Walking a prompt through the decode step reads every dense weight, the picked
experts and the whole recurrent state once per token, and the head for logits nobody
reads.  A pass takes up to ``MAX_PASS`` rows -- T consecutive tokens of each of the
engine's sequences -- through each layer (``csrc/prefill_hybrid.hip``): projections
and experts for all rows together, attention over the paged cache, and only the
recurrence token by token, its state in registers.  Each row is valued as a step at
its position values it, with f32 sums in other orders, and Granite's attention takes
exact products and rounds each probability against the maximum so far (a step rounds
the products and the normalised probabilities).

The pass leaves what the walk leaves for the next step: caches, recurrent states and
convolution windows of positions 0 .. n - 2.  So the last layer stops at its mixer's
state (or its keys and values); nothing reads what would follow.
"""
from __future__ import annotations

import ctypes
import weakref

import numpy as np
import torch

from .. import _lib
from .._lib import lib, ptr
from ..qwen3.prefill import plan_passes, token_array, wait_for_work

MAX_PASS = 1024             # rows of one pass: its workspaces take up to about 0.4 GB

BF, F32, I32 = torch.bfloat16, torch.float32, torch.int32


def _addr(struct) -> int:
    return ctypes.addressof(struct)


class _Pass:
    """What both models' passes share: *eng* is the engine; subclasses give the
    layer's shape and mixer."""

    policy: int
    fp8: bool

    @staticmethod
    def step_positions(seqs: int) -> int:
        """Positions per sequence up to which the decode step's walk is as fast."""
        return 1

    def __init__(self, eng):
        # the engine holds this pass: a strong reference back would keep both, and
        # their device memory, until a garbage collection
        self._eng, self.cfg, self._lib = weakref.ref(eng), eng.cfg, lib()
        self.B, self.H, self.k = eng.B, eng.cfg.hidden, eng.cfg.top_k
        self.dev = eng.device
        self.layers = [self._weights(w) for w in eng.layers]
        torch.cuda.synchronize(self.dev)
        self.rows = 0

    @property
    def e(self):
        return self._eng()

    def _stream(self) -> int:
        return torch.cuda.current_stream(self.dev).cuda_stream

    def _reserve(self, M):
        if M <= self.rows:
            return
        R = -(-M // 32) * 32
        if self.rows:
            wait_for_work(self.dev)
        self.rows = 0                       # until every buffer below holds R rows
        c, H, k = self.cfg, self.H, self.k
        shapes = [(H, self.in_rows), (self.out_k, H), (H, c.experts), (H, 2 * c.shared_inter),
                  (c.shared_inter, H)]
        if self.attn_k:
            shapes += [(self.attn_k, H), (H, c.attn_in)]
        part = max(self._lib.tfd_panel_gemm_slices(m, K, N) * m * N
                   for K, N in shapes for m in range(32, R + 1, 32))

        def z(*shape, dtype=BF):
            return torch.zeros(*shape, device=self.dev, dtype=dtype)

        self.nproj = -(-max(self.in_rows, c.attn_in) // 8) * 8
        self.part = z(part, dtype=F32)
        self.emb, self.xm, self.xn = z(R, H), z(R, H), z(R * H)
        self.proj, self.mix = z(R, self.nproj), z(R * max(self.out_k, self.attn_k))
        self.rlog, self.rw = z(R, c.experts, dtype=F32), z(R, k, dtype=F32)
        self.ridx = z(R, k, dtype=I32)
        self.groups = z(_lib.panel_moe_words(c.experts, R * k), dtype=I32)
        self.moe_hidden, self.d = z(R * k, c.moe_inter), z(R * k, H)
        self.shared = z(R * c.shared_inter)
        self._mixer_buffers(R, z)
        self.rows = R

    # ------------------------------------------------------------------ pieces
    def _gemm(self, x, w, scale, M, K, N, s):
        """K-split partial sums of x @ w^T in ``part`` -> their number."""
        if self.fp8:
            self._lib.tfd_panel_gemm_fp8(ptr(x), ptr(w), ptr(scale), M, K, N, ptr(self.part), s)
        else:
            self._lib.tfd_panel_gemm_bf16(ptr(x), ptr(w), M, K, N, _lib.PANEL_PARTIAL,
                                          ptr(self.part), s)
        return self._lib.tfd_panel_gemm_slices(M, K, N)

    def _update(self, M, slices, gamma, s, *, rows=False, moe=None):
        """The stream plus ``part``'s sums (with *moe*, the experts' mix), and the
        norm by *gamma* into xn (and the row-major xm)."""
        a = _lib.TfdPanelMixArgs()
        a.part, a.slices, a.stream_rows = ptr(self.part), slices, ptr(self.stream)
        a.mult, a.M, a.n, a.policy, a.eps = self.mult, M, self.H, self.policy, self.cfg.eps
        if moe is not None:
            a.moe, a.k, a.d, a.weights = 1, self.k, ptr(self.d), ptr(self.rw)
            a.x_moe, a.w_shared_scale = ptr(self.xm), ptr(moe.get("w_shared_scale"))
        a.gamma, a.norm_panels = ptr(gamma), ptr(self.xn)
        a.norm_rows = ptr(self.xm) if rows else None
        self._lib.tfd_panel_mix(_addr(a), s)

    def _attention(self, i, w, M, at, tiles, s):
        e, c = self.e, self.cfg
        a = _lib.TfdPanelGqaArgs()
        a.proj, a.ldp, a.M, a.policy, a.err = ptr(self.proj), self.nproj, M, self.policy, \
            ptr(e.err)
        a.pos, a.seq, a.tiles, a.ntiles = at + 4 * M, at + 8 * M, at + 12 * M, tiles
        a.page_table, a.max_pages, a.num_pages = ptr(e.page_table), e.max_pages, e.num_pages
        a.k_pool, a.v_pool = ptr(e.kpool[i]), ptr(e.vpool[i])
        a.heads, a.kv_heads, a.head_dim, a.eps = c.heads, c.kv_heads, c.head_dim, c.eps
        a.q, a.out = ptr(self.q), ptr(self.mix)
        self._attention_args(a, w)
        self._lib.tfd_panel_gqa(_addr(a), s)

    def _moe(self, w, M, s):
        """The routed experts' outputs in ``d`` and the shared expert's sums in
        ``part`` -> their slices."""
        c, L, H = self.cfg, self._lib, self.H
        sl = self._gemm(self.xn, w["w_router"], w.get("w_router_scale"), M, H, c.experts, s)
        L.tfd_panel_sum(ptr(self.part), sl, M, c.experts, ptr(self.rlog), c.experts, 1, s)
        L.tfd_route_topk(ptr(self.rlog), c.experts, M, c.experts, self.k, self.route,
                         ptr(self.rw), ptr(self.ridx), s)
        a = _lib.TfdPanelMoeArgs()
        a.x, a.idx, a.groups = ptr(self.xm), ptr(self.ridx), ptr(self.groups)
        a.w_gate, a.w_up, a.w_down = ptr(w["w_gate"]), ptr(w["w_up"]), ptr(w["w_down"])
        a.s_gate, a.s_up, a.s_down = ptr(w.get("s_gate")), ptr(w.get("s_up")), \
            ptr(w.get("s_down"))
        a.hidden, a.d, a.err = ptr(self.moe_hidden), ptr(self.d), ptr(self.e.err)
        a.M, a.k, a.experts, a.H, a.I = M, self.k, c.experts, H, c.moe_inter
        a.fp8, a.policy = int(self.fp8), self.policy
        L.tfd_panel_moe(_addr(a), s)
        IS = c.shared_inter
        sl = self._gemm(self.xn, w["p_shared_in"], w.get("w_shared_in_scale"), M, H, 2 * IS, s)
        L.tfd_panel_swiglu_halves(ptr(self.part), sl, M, 2 * IS, self.policy, ptr(self.shared), s)
        return self._gemm(self.shared, w["p_shared_out"], w.get("w_shared_out_scale"), M, IS, H,
                          s)

    def _layer(self, i, T, M, at, tiles, cur, s):
        w, full = self.layers[i], self._is_full(i)
        N = self.cfg.attn_in if full else self.in_rows
        sl = self._gemm(self.xn, w["w_in"], w.get("w_in_scale"), M, self.H, N, s)
        self._lib.tfd_panel_sum(ptr(self.part), sl, M, N, ptr(self.proj), self.nproj, 0, s)
        if full:
            self._attention(i, w, M, at, tiles, s)
        else:
            self._mixer(i, w, T, cur, s)
        if i + 1 == self.cfg.layers:
            return
        sl = self._gemm(self.mix, w["w_out"], w.get("w_out_scale"), M,
                        self.attn_k if full else self.out_k, self.H, s)
        self._update(M, sl, w["gamma_post"], s, rows=True)
        sl = self._moe(w, M, s)
        self._update(M, sl, self.layers[i + 1]["gamma_in"], s, moe=w)

    def run(self, prompts: list[list[int]]):
        """Positions 0 .. n - 2 of every sequence (prompts of one length n), from the
        engine's state as ``_load_prompts`` leaves it."""
        e, n = self.e, len(prompts[0]) - 1
        prompts = [token_array(p) for p in prompts]
        span = max(1, MAX_PASS // self.B)
        for t0 in range(0, n, span):
            T = min(span, n - t0)
            M = self.B * T
            self._reserve(M)
            segments = [(p[t0:t0 + T], t0, b) for b, p in enumerate(prompts)]
            (ids, pos, seqs, tiles), = plan_passes(segments, M, self.tile_rows)
            flat = torch.from_numpy(np.concatenate((ids, pos, seqs, tiles.reshape(-1)))).to(
                self.dev)
            token = flat[:M].to(torch.int64)
            s = self._stream()
            self._lib.tfd_embed_rows_bf16(ptr(e.embed), ptr(token), ptr(self.emb), self.H, M,
                                          self.H, self.cfg.vocab, ptr(e.err), s)
            self._start(M, s)
            self._update(M, 0, self.layers[0]["gamma_in"], s)
            for i in range(self.cfg.layers):
                self._layer(i, T, M, ptr(flat), len(tiles), e._cur, s)
            e._cur ^= 1


class Qwen35Pass(_Pass):
    """Qwen3.5: f32 stream, gated DeltaNet, bf16 weights."""

    policy, fp8, mult = _lib.POLICY_F32, False, 1.0
    route, tile_rows = _lib.ROUTE_SOFTMAX_TOPK, _lib.PANEL_GQA_ROWS_F32

    def __init__(self, eng):
        c = eng.cfg
        self.in_rows, self.out_k = c.gdn_in, c.value_dim
        self.attn_k = c.heads * c.head_dim
        super().__init__(eng)

    @staticmethod
    def step_positions(seqs: int) -> int:
        # four layers: one sequence's two positions 604 us walked, 691 in a pass, three
        # 829 / 682; two sequences' two positions 774 / 722, sixteen's 1,886 / 1,587
        return 2 if seqs == 1 else 1

    @staticmethod
    def takes(eng) -> bool:
        """Whether the kernels of a pass cover this engine's sizes."""
        c = eng.cfg
        ks = (c.hidden, c.value_dim, c.heads * c.head_dim, c.shared_inter)
        return (c.lin_key_dim == c.lin_value_dim == 128 and c.conv_kernel == 4 and
                c.lin_value_heads % c.lin_key_heads == 0 and all(k % 256 == 0 for k in ks) and
                c.hidden <= 8192 and c.moe_inter % 128 == 0 and c.experts <= 256 and
                c.experts % 4 == 0 and c.gdn_in % 4 == 0 and c.head_dim == 256 and
                c.heads == 8 * c.kv_heads)

    def _packed(self, w):
        N, K = w.shape
        out = torch.empty(-(-N // 16) * 16 * K, dtype=BF, device=self.dev)
        self._lib.tfd_pack_skinny_bf16(ptr(w), K, N, K, ptr(out), self._stream())
        return out

    def _weights(self, w):
        """The layer's matrices in the panel GEMMs' blocks: the batched engine's
        projections as they are, a copy of the small-batch engine's rows."""
        w = dict(w)
        if self.e.small:
            for n in ("w_in", "w_out", "w_router"):
                w[n] = self._packed(w[n])
        w["p_shared_in"] = self._packed(w["w_shared_in"])
        w["p_shared_out"] = self._packed(w["w_shared_out"])
        return w

    def _is_full(self, i):
        return self.cfg.is_full(i)

    def _mixer_buffers(self, R, z):
        c = self.cfg
        self.stream = z(R, self.H, dtype=F32)
        self.qk, self.v = z(2 * R * c.key_dim, dtype=F32), z(R * c.value_dim, dtype=F32)
        self.read = z(R * c.value_dim, dtype=F32)
        self.gates = z(R * c.lin_value_heads * 2, dtype=F32)
        self.q, self.gate = z(R * self.attn_k, dtype=F32), z(R * self.attn_k)
        self.self_scores = z(R * c.heads, dtype=F32)

    def _start(self, M, s):
        self._lib.tfd_bf16_to_f32_rows(ptr(self.emb), self.H, ptr(self.stream), self.H, M, self.H,
                                       s)

    def _attention_args(self, a, w):
        e, c = self.e, self.cfg
        a.gamma_q, a.gamma_k = ptr(w["gamma_q"]), ptr(w["gamma_k"])
        a.cos_table, a.sin_table = ptr(e.cos), ptr(e.sin)
        a.rope_rows, a.rot_dim, a.scale = e.cos.shape[0], c.rot_dim, c.head_dim ** -0.5
        a.gate, a.self_scores = ptr(self.gate), ptr(self.self_scores)

    def _mixer(self, i, w, T, cur, s):
        e, c = self.e, self.cfg
        a = _lib.TfdPanelGdnArgs()
        a.proj, a.ldp, a.seqs, a.T = ptr(self.proj), self.nproj, self.B, T
        a.conv_in, a.conv_out = ptr(e.conv[i][cur]), ptr(e.conv[i][1 - cur])
        a.state, a.conv_w, a.a_log = ptr(e.state[i]), ptr(w["conv_w"]), ptr(w["a_log"])
        a.dt_bias, a.gamma = ptr(w["dt_bias"]), ptr(w["gamma_gdn"])
        a.qk, a.v, a.read, a.gates = ptr(self.qk), ptr(self.v), ptr(self.read), ptr(self.gates)
        a.out, a.key_heads, a.value_heads = ptr(self.mix), c.lin_key_heads, c.lin_value_heads
        a.head_dim, a.l2_eps, a.rms_eps = c.lin_key_dim, 1e-6, c.eps
        self._lib.tfd_panel_gdn(_addr(a), s)


class GranitePass(_Pass):
    """Granite-4.0-H: bf16 stream, Mamba2, fp8 weights packed for the matrix cores."""

    policy, fp8 = _lib.POLICY_BF16, True
    route, tile_rows = _lib.ROUTE_TOPK_SOFTMAX, _lib.PANEL_GQA_ROWS_BF16

    def __init__(self, eng):
        c = eng.cfg
        self.in_rows, self.out_k = c.mamba_in, c.d_inner
        self.attn_k = c.heads * c.head_dim
        self.mult = c.residual_multiplier
        super().__init__(eng)

    @staticmethod
    def takes(eng) -> bool:
        """Whether the kernels of a pass cover this engine's sizes and weights."""
        c = eng.cfg
        ks = (c.hidden, c.d_inner, c.heads * c.head_dim, c.shared_inter)
        return (eng.moe_packed and c.mamba_head_dim == 64 and c.d_state == 128 and
                c.conv_kernel == 4 and all(k % 256 == 0 for k in ks) and c.hidden <= 8192 and
                c.d_inner <= 8192 and c.moe_inter % 128 == 0 and c.experts <= 256 and
                c.experts % 4 == 0 and c.mamba_in % 4 == 0 and c.head_dim == 128 and
                c.heads == 4 * c.kv_heads)

    def _weights(self, w):
        w = dict(w)
        w["p_shared_in"], w["p_shared_out"] = w["w_shared_in"], w["w_shared_out"]
        return w

    def _is_full(self, i):
        return self.cfg.is_attention(i)

    def _mixer_buffers(self, R, z):
        c = self.cfg
        self.stream = z(R, self.H)
        self.x, self.y = z(R * c.d_inner), z(R * c.d_inner)
        self.bc, self.gates = z(R * 2 * c.d_state), z(R * c.mamba_heads * 2, dtype=F32)
        self.q = z(R * self.attn_k)

    def _start(self, M, s):
        self._lib.tfd_scaled_add_rows(None, 0, ptr(self.emb), self.H, 0,
                                      self.cfg.embedding_multiplier, ptr(self.stream), self.H, M,
                                      self.H, s)

    def _attention_args(self, a, w):
        a.scale = self.cfg.attention_multiplier

    def _mixer(self, i, w, T, cur, s):
        e, c = self.e, self.cfg
        a = _lib.TfdPanelMambaArgs()
        a.proj, a.ldp, a.seqs, a.T = ptr(self.proj), self.nproj, self.B, T
        a.conv_in, a.conv_out = ptr(e.conv[i][cur]), ptr(e.conv[i][1 - cur])
        a.state, a.conv_w, a.conv_b = ptr(e.state[i]), ptr(w["conv_w"]), ptr(w["conv_b"])
        a.a_log, a.dt_bias, a.d_skip = ptr(w["a_log"]), ptr(w["dt_bias"]), ptr(w["d_skip"])
        a.gamma, a.x, a.bc, a.y = ptr(w["gamma_ssm"]), ptr(self.x), ptr(self.bc), ptr(self.y)
        a.gates, a.out, a.heads = ptr(self.gates), ptr(self.mix), c.mamba_heads
        a.head_dim, a.state_dim, a.eps = c.mamba_head_dim, c.d_state, c.eps
        self._lib.tfd_panel_mamba(_addr(a), s)


def prefill(eng, passes, prompts: list[list[int]]):
    """Bring *eng* to every prompt's last token: passes of class *passes* where their
    kernels take the engine's sizes, else the decode step walked position by position.
    (A pass leaves no routing and no logits of the prompt's own positions.)"""
    if len(prompts) != eng.B or any(len(p) < 1 for p in prompts):
        raise ValueError(f"need {eng.B} non-empty prompts")
    if len({len(p) for p in prompts}) != 1:
        raise ValueError("prefill: the prompts must have one length (the walk moves "
                         "every sequence one position per step)")
    n = len(prompts[0])
    if n > eng.nsteps:
        raise ValueError(f"prompt {n} exceeds {eng.nsteps} steps")
    eng._load_prompts(prompts)
    # One position: a step's kernels, made for a row a sequence, are faster than a pass
    # (four layers, one sequence: Qwen3.5 319 against 577 us, Granite 449 / 628; two
    # positions of Granite 813 / 648; of Qwen3.5 see its ``step_positions``).
    # An engine that records its routing keeps the last walked position's.
    walk = n - 1 <= passes.step_positions(eng.B) or eng.routes is not None
    if walk or not passes.takes(eng):
        for _ in range(n - 1):
            eng.replay()
        return
    if getattr(eng, "_prefiller", None) is None:
        eng._prefiller = passes(eng)
    eng._prefiller.run(prompts)
    eng.pos.fill_(n - 1)
    eng.ids.copy_(torch.tensor([p[-1] for p in prompts], dtype=torch.int64))
    eng._lib.tfd_embed_rows_bf16(ptr(eng.embed), ptr(eng.ids), ptr(eng.emb), eng.cfg.hidden,
                                 eng.B, eng.cfg.hidden, eng.cfg.vocab, ptr(eng.err),
                                 eng._stream())
