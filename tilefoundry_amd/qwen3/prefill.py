"""Prompt prefill: a prompt's positions through every layer together.

The reference's engine walks a prompt one token per replayed decode step
(``examples/qwen3_1_7b-tilelang/fast/engine.py:261-262``); its placed fixture
``tests/fixtures/placed/qwen3_1_7b_pd.py:55-230`` (``layer_prefill``) is the
batched form: the prompt rows go through the norm, one q/k/v GEMM, q/k norm +
RoPE, the cache update for every row, causal attention and the MLP GEMMs
together.  Here a pass takes up to ``MAX_PASS`` rows, of one or of several
sequences, through each layer (``csrc/prefill.hip``): every weight is read once per
pass and every cached key once per 64 rows of a tile, where the decode kernels
would read them once per 32 rows and once per row.  Each position is valued as a
decode step at that position values it: the HIR's rounding points, with attention's
products exact as the XCD kernel takes them, each probability rounded against the
maximum of the tiles so far, and other f32 summation orders.

Prefill fills the cache for positions start .. start + n - 1 and leaves the
hidden states of those rows unused: the last prompt token is then decoded as
before, by the decode step, which produces the first new token.  So the last layer
stops at its keys and values; nothing reads what would follow.

The same pass serves a batch engine (``batch_engine.py``): its sequences share
one pool of pages, each with its own page-table row, and the prompts of all of them
go through together.
"""
from __future__ import annotations

import weakref
from array import array
from operator import index

import numpy as np
import torch

from .. import _lib
from .._lib import lib, ptr

MAX_PASS = 4096             # rows of one pass: its workspaces take about 0.3 GB

# The batched attention's grid is (splits, kv heads, rows): about two blocks per
# compute unit (256 on the MI355X) keeps every split long enough that its tiles
# stream back to back.  At batch 32 over 4,159 positions, measured per layer:
# scores + P.V 98.8 us with 2 splits, 99.8 with 3, 102.8 with 4, 111.7 with 17.
SPLIT_BLOCKS = 512


def attention_splits(rows: int, kv_heads: int, cap: int) -> int:
    """Splits per (row, kv head) of the batched attention for *rows* rows; their
    length follows each row's position (``split_tiles`` 0)."""
    tiles = -(-cap // _lib.ATTN_SPLIT)
    return max(1, min(tiles, -(-SPLIT_BLOCKS // (rows * kv_heads))))


def gate_up_panels(rows: int, inter: int, cus: int) -> bool:
    """Whether the gate/up projection of *rows* rows goes through the panel GEMM rather
    than the skinny one (which takes up to 32).  The panel GEMM multiplies 32 rows
    whatever their number, the skinny one 16 up to 16; and its blocks of 64 columns want
    full rounds of the *cus* compute units.  Steps of three or four layers with the skinny
    / the panel gate/up (hidden x inter, us): 16 rows 2,048 x 6,144 216 / 219, 4,096 x
    12,288 (1.5 rounds of blocks) 297 / 320, 2,560 x 9,728 (1.2 rounds) 289 / 341; 24 rows
    226 / 221, 318 / 325, 317 / 344; 32 rows 240 / 231, 343 / 335, 341 / 354."""
    if rows <= 16 or rows > 32:
        return rows > 32
    blocks = -(-2 * inter // 64)
    return 10 * blocks >= 7 * cus * -(-blocks // cus)


def token_array(tokens) -> np.ndarray:
    """Token ids (any sequence of them) as an int64 array."""
    try:
        if isinstance(tokens, (list, tuple)):
            try:                            # whole numbers, tensors of one element too
                return np.array(array("q", tokens))
            except TypeError:               # fractions are cut, as int() cuts them
                return np.array([int(t) if isinstance(t, (float, np.floating, torch.Tensor))
                                 else index(t) for t in tokens], dtype=np.int64)
        if isinstance(tokens, torch.Tensor):
            tokens = tokens.detach().cpu()
            tokens = tokens.double() if tokens.is_floating_point() else tokens
        ids = np.asarray(tokens)
        if ids.ndim != 1 or ids.dtype.kind not in "biuf":
            raise TypeError
    except OverflowError:
        raise ValueError("token ids must fit in 64 bits") from None
    except TypeError:
        raise ValueError("token ids must be one sequence of whole numbers") from None
    if ids.dtype.kind == "f" and not (np.abs(ids) < 2.0 ** 63).all():
        raise ValueError("token ids must fit in 64 bits")
    return ids.astype(np.int64, copy=False)


def int32_ids(tokens) -> np.ndarray:
    """``token_array`` as the int32 values the device buffers hold."""
    ids = token_array(tokens)
    if not in_vocab(np.abs(ids), 1 << 31):
        raise RuntimeError("token ids must fit in 32 bits")
    return ids.astype(np.int32)


def wait_for_work(device):
    """Wait for the current stream, before buffers go that launches on it may still use:
    the allocator hands a freed block on at once to the stream that allocated it, which
    need not be this one."""
    torch.cuda.current_stream(device).synchronize()


def in_vocab(tokens: np.ndarray, vocab: int) -> bool:
    return tokens.size == 0 or (int(tokens.min()) >= 0 and int(tokens.max()) < vocab)


def plan_passes(segments, max_rows: int, tile_rows: int):
    """Cut (tokens, start, seq) segments into passes of at most *max_rows* rows ->
    per pass (ids, pos, seq, tiles), int32 arrays: the token, position and sequence of
    each row, and the attention tiles [n][4] (first row, rows, sequence, first position),
    the deepest first (they take longest, so none of them is left to the end of a
    launch)."""
    passes, parts, rows = [], [], 0

    def close():
        nonlocal parts, rows
        if parts:
            ids = np.concatenate([t for t, _, _ in parts]).astype(np.int32)
            pos = np.concatenate([np.arange(p, p + len(t), dtype=np.int32) for t, p, _ in parts])
            seqs = np.concatenate([np.full(len(t), q, dtype=np.int32) for t, _, q in parts])
            tiles, row0 = [], 0
            for t, p, q in parts:
                at = np.arange(0, len(t), tile_rows, dtype=np.int32)
                tiles.append(np.stack((row0 + at, np.minimum(tile_rows, len(t) - at),
                                       np.full_like(at, q), p + at), axis=1))
                row0 += len(t)
            tiles = np.concatenate(tiles)
            tiles = tiles[np.argsort(-(tiles[:, 3] + tiles[:, 1]), kind="stable")]
            passes.append((ids, pos, seqs, tiles.astype(np.int32)))
        parts, rows = [], 0

    for tokens, start, seq in segments:
        tokens, done = token_array(tokens), 0
        while done < len(tokens):
            n = min(len(tokens) - done, max_rows - rows)
            if n == 0:
                close()
                continue
            parts.append((tokens[done:done + n], start + done, seq))
            rows += n
            done += n
    close()
    return passes


class Prefill:
    """The batched prompt pass over an engine's weights, pools and page table.

    *engine* is a ``qwen3.engine.Engine`` (or anything with its attributes:
    ``layers``, ``kpool``/``vpool`` [L][pages][HKV][16][D], ``page_table``
    ([max_pages], or [sequences][max_pages] with ``num_pages`` pages in the
    pool), ``cos``/``sin``, ``cap``).  With *packed* False the projections are
    re-laid once into the skinny GEMMs' operand blocks (one more copy of the
    layer weights in HBM); a batch engine's layers are already in that order.
    An engine that keeps its own pass hands in a weak reference to itself: with a cycle the
    device memory of both would stay until a garbage collection.  Workspaces grow to the
    largest pass seen, ``MAX_PASS`` rows at most."""

    def __init__(self, engine, packed: bool = False):
        self._engine = engine if isinstance(engine, weakref.ref) else lambda: engine
        e = self.e
        self._lib = lib()
        self.dev = e.device
        self.L, self.H, self.I, self.D = e.L, e.H, e.I, e.D
        self.HQ, self.HKV = e.HQ, e.HKV
        self.QD = self.HQ * self.D
        self.qkv_n = e.cfg.qkv_size
        self.eps, self.scale = e.eps, e.scale
        self.max_pages = e.max_pages
        self.num_pages = getattr(e, "num_pages", e.max_pages)
        self.seqs = e.page_table.numel() // self.max_pages
        self.tile_rows = self._lib.tfd_panel_attn_rows(self.HQ // self.HKV)
        s = torch.cuda.current_stream(self.dev).cuda_stream
        self.layers = []
        for w in e.layers:
            lw = dict(w)
            if not packed:
                for n in ("w_qkv", "w_o", "w_gu", "w_down"):
                    lw[n] = self._mfma_order(w[n], s)
            self.layers.append(lw)
        # the skinny GEMM's tile counters (kept at zero by the library) and partial tiles
        self.work = torch.zeros(1 << 21, device=self.dev, dtype=torch.float32)
        self.cus = torch.cuda.get_device_properties(self.dev).multi_processor_count
        torch.cuda.synchronize(self.dev)
        self.rows = 0

    @property
    def e(self):
        return self._engine()

    def _mfma_order(self, w, s):
        N, K = w.shape
        out = torch.empty(-(-N // 16) * 16, K, device=w.device, dtype=w.dtype)
        self._lib.tfd_pack_skinny_bf16(ptr(w), K, N, K, ptr(out), s)
        return out

    def _slices(self, M, K, N):
        return self._lib.tfd_panel_gemm_slices(M, K, N)

    def _reserve(self, M):
        """Workspaces for passes of up to M rows."""
        if M <= self.rows:
            return
        R = -(-M // 32) * 32
        if self.rows:
            wait_for_work(self.dev)
        self.rows = 0                       # until every buffer below holds R rows
        dev, bf, f32 = self.dev, torch.bfloat16, torch.float32
        shapes = [(self.H, self.qkv_n), (self.QD, self.H), (self.I, self.H), (self.H, 2 * self.I)]
        part = 1
        for K, N in shapes:
            for m in range(32, R + 1, 32):
                sl = self._slices(m, K, N)
                if N != 2 * self.I or sl > 1:      # gate/up: only its K splits leave partials
                    part = max(part, sl * m * N)
        self.hid = torch.empty(R, self.H, device=dev, dtype=bf)
        self.h1 = torch.empty(R, self.H, device=dev, dtype=bf)
        self.xn = torch.zeros(R * self.H, device=dev, dtype=bf)
        self.q = torch.empty(R, self.QD, device=dev, dtype=bf)
        self.attn = torch.zeros(R * self.QD, device=dev, dtype=bf)
        self.hmid = torch.zeros(R * self.I, device=dev, dtype=bf)
        self.part = torch.empty(part, device=dev, dtype=f32)
        self.rows = R

    def _gemm(self, x, w, M, K, N, s):
        """K-split partial sums of x @ w^T -> their number."""
        self._lib.tfd_panel_gemm_bf16(ptr(x), ptr(w), M, K, N, _lib.PANEL_PARTIAL, ptr(self.part),
                                      s)
        return self._slices(M, K, N)

    def _layer(self, i, M, pos, seq, tiles, ntiles, s):
        """One decoder layer (model.py:236-266) for M prompt rows; xn holds its
        normalised input.  The last layer stops at its keys and values."""
        L, w, e = self._lib, self.layers[i], self.e
        H, I = self.H, self.I
        table = ptr(e.page_table)
        sl = self._gemm(self.xn, w["w_qkv"], M, H, self.qkv_n, s)
        L.tfd_panel_qkv_append(
            ptr(self.part), sl, M, self.HQ, self.HKV, self.D, ptr(w["gamma_q"]),
            ptr(w["gamma_k"]), ptr(e.cos), ptr(e.sin), e.cap, pos, seq, table, self.max_pages,
            ptr(e.kpool[i]), ptr(e.vpool[i]), self.num_pages, self.scale, self.eps, ptr(self.q),
            ptr(e.err), s)
        if i + 1 == self.L:
            return
        L.tfd_panel_attn(ptr(self.q), tiles, ntiles, self.HQ, self.HKV, self.D, table,
                         self.max_pages, ptr(e.kpool[i]), ptr(e.vpool[i]), self.num_pages,
                         ptr(self.attn), ptr(e.err), s)
        sl = self._gemm(self.attn, w["w_o"], M, self.QD, H, s)
        L.tfd_panel_add_norm(ptr(self.part), sl, ptr(self.hid), ptr(self.h1),
                             ptr(w["gamma_post"]), ptr(self.xn), M, H, self.eps, s)
        slices = self._slices(M, H, 2 * I)
        if M <= 16 or not (slices > 1 or gate_up_panels(M, I, self.cus)):
            L.tfd_gemm_skinny_bf16(ptr(self.xn), ptr(w["w_gu"]), M, H, 2 * I, _lib.EPI_SWIGLU,
                                   None, 0, ptr(self.hmid), 0, ptr(self.work),
                                   self.work.numel(), s)
        elif slices == 1:
            L.tfd_panel_gemm_bf16(ptr(self.xn), ptr(w["w_gu"]), M, H, 2 * I, _lib.PANEL_SWIGLU,
                                  ptr(self.hmid), s)
        else:
            sl = self._gemm(self.xn, w["w_gu"], M, H, 2 * I, s)
            L.tfd_panel_swiglu(ptr(self.part), sl, M, 2 * I, ptr(self.hmid), s)
        sl = self._gemm(self.hmid, w["w_down"], M, I, H, s)
        L.tfd_panel_add_norm(ptr(self.part), sl, ptr(self.h1), ptr(self.hid),
                             ptr(self.layers[i + 1]["gamma_in"]), ptr(self.xn), M, H, self.eps, s)

    def run(self, tokens: list[int], start: int = 0, seq: int = 0):
        """Fill every layer's cache at positions start .. start + len(tokens) - 1
        of sequence *seq* (its page-table row) from those tokens."""
        self.run_many([(tokens, start, seq)])

    def run_many(self, segments):
        """``run`` for several (tokens, start, seq) at once; a sequence's segments in
        the order of their positions."""
        e = self.e
        for tokens, start, seq in segments:
            if start < 0 or start + len(tokens) > e.cap:
                raise ValueError(f"prefill: positions {start}..{start + len(tokens) - 1} outside "
                                 f"the cache ({e.cap} positions)")
            if not in_vocab(token_array(tokens), e.V):
                raise ValueError(f"prefill: token ids must lie in [0, {e.V})")
            if not 0 <= seq < self.seqs:
                raise ValueError(f"prefill: sequence {seq} outside [0, {self.seqs})")
        s = torch.cuda.current_stream(self.dev).cuda_stream
        for ids, pos, seqs, tiles in plan_passes(segments, MAX_PASS, self.tile_rows):
            M = len(ids)
            self._reserve(M)
            flat = torch.from_numpy(np.concatenate((ids, pos, seqs, tiles.reshape(-1)))).to(
                self.dev)
            at = ptr(flat)
            token = flat[:M].to(torch.int64)
            self._lib.tfd_embed_rows_bf16(ptr(e.w_embed), ptr(token), ptr(self.hid), self.H, M,
                                          self.H, e.V, ptr(e.err), s)
            self._lib.tfd_panel_add_norm(None, 0, ptr(self.hid), None,
                                         ptr(self.layers[0]["gamma_in"]), ptr(self.xn), M, self.H,
                                         self.eps, s)
            for i in range(self.L):
                self._layer(i, M, at + 4 * M, at + 8 * M, at + 12 * M, len(tiles), s)
