"""Prompt-pass kernels (csrc/prefill.hip) against plain f32 references, at the
sizes where tiles and passes end, and the cut of prompts into passes (CPU)."""
import ctypes

import pytest
import torch

from tilefoundry_amd import _lib
from tilefoundry_amd.qwen3.prefill import plan_passes


def panels(x):
    """[M][K] rows in panel order (32-row panels in operand order, zero padded)."""
    M, K = x.shape
    P = -(-M // 32)
    z = torch.zeros(P * 32, K, device=x.device, dtype=x.dtype)
    z[:M] = x
    return z.view(P, 2, 16, K // 32, 4, 8).permute(0, 3, 1, 4, 2, 5).contiguous().reshape(-1)


def unpanel(flat, M, K):
    P = -(-M // 32)
    return flat[:P * 32 * K].view(P, K // 32, 2, 4, 16, 8).permute(0, 2, 4, 1, 3, 5).reshape(
        P * 32, K)[:M]


@pytest.mark.parametrize("lens,max_rows,tile", [
    ([1], 4096, 64), ([64, 65, 1], 4096, 64), ([130, 7, 300], 100, 64), ([33, 33, 33], 32, 128),
])
def test_plan_passes_covers_every_row_once(lens, max_rows, tile):
    segments = [([1000 * b + i for i in range(n)], 5 * b, b) for b, n in enumerate(lens)]
    seen = []
    for plan in plan_passes(segments, max_rows, tile):
        ids, pos, seqs, tiles = (a.tolist() for a in plan)
        assert 0 < len(ids) <= max_rows and len(ids) == len(pos) == len(seqs)
        rows = []
        for row0, n, seq, p0 in tiles:
            assert 0 < n <= tile
            assert seqs[row0:row0 + n] == [seq] * n
            assert pos[row0:row0 + n] == list(range(p0, p0 + n))
            rows += range(row0, row0 + n)
        assert sorted(rows) == list(range(len(ids)))
        assert [t[3] + t[1] for t in tiles] == sorted((t[3] + t[1] for t in tiles), reverse=True)
        seen += list(zip(seqs, pos, ids))
    # each sequence's rows in the order of its positions, every one once
    for b, (tokens, start, _) in enumerate(segments):
        mine = [(p, t) for s, p, t in seen if s == b]
        assert mine == [(start + i, t) for i, t in enumerate(tokens)]


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 31, 33, 64, 97, 128, 129, 300, 1100])
@pytest.mark.parametrize("K,N", [(256, 768), (768, 256), (2048, 1056), (6144, 2048), (512, 40)])
def test_panel_gemm(gpu_device, M, K, N):
    """f32 sums of exact bf16 products: |error| <= K 2^-24 sum|x w| for any order."""
    L = _lib.lib()
    s = torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=gpu_device).manual_seed(M * 7 + K)
    x = torch.randn(M, K, generator=g, device=gpu_device).to(torch.bfloat16)
    w = torch.randn(N, K, generator=g, device=gpu_device).to(torch.bfloat16)
    packed = torch.empty(-(-N // 16) * 16 * K, device=gpu_device, dtype=torch.bfloat16)
    L.tfd_pack_skinny_bf16(w.data_ptr(), K, N, K, packed.data_ptr(), s)
    xp = panels(x)
    slices = L.tfd_panel_gemm_slices(M, K, N)
    assert slices >= 1 and (K // 32) % slices == 0
    part = torch.full((slices, M, N), float("nan"), device=gpu_device)
    L.tfd_panel_gemm_bf16(xp.data_ptr(), packed.data_ptr(), M, K, N, _lib.PANEL_PARTIAL,
                          part.data_ptr(), s)
    want = x.double() @ w.double().t()
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert ((part.double().sum(0) - want).abs() <= bound).all()
    if N % 64:
        return
    # SwiGLU, from the partial sums (added in slice order, as the kernel adds them) and
    # (one slice) from the GEMM itself: two bf16 roundings after the sums, which an ulp
    # of exp may settle another way
    r = part[0].clone()
    for sl in range(1, slices):
        r += part[sl]
    r = r.to(torch.bfloat16).float()
    act = torch.nn.functional.silu(r[:, 0::2]).to(torch.bfloat16).float() * r[:, 1::2]
    out = torch.zeros(-(-M // 32) * 32 * (N // 2), device=gpu_device, dtype=torch.bfloat16)
    L.tfd_panel_swiglu(part.data_ptr(), slices, M, N, out.data_ptr(), s)
    assert ((unpanel(out, M, N // 2).float() - act).abs() <= 2.0 ** -6 * act.abs() + 1e-6).all()
    if slices == 1:
        two = torch.zeros_like(out)
        L.tfd_panel_gemm_bf16(xp.data_ptr(), packed.data_ptr(), M, K, N, _lib.PANEL_SWIGLU,
                              two.data_ptr(), s)
        assert torch.equal(two, out)


@pytest.mark.gpu
@pytest.mark.parametrize("slices,M,n", [(0, 1, 256), (1, 33, 2048), (3, 65, 2048), (2, 5, 4096)])
def test_panel_add_norm(gpu_device, slices, M, n):
    """The residual sum rounds once more (equal bits: the slices add in order); the
    norm is bf16(bf16(h r) gamma), r within f32 rounding: one ulp of either."""
    L = _lib.lib()
    g = torch.Generator(device=gpu_device).manual_seed(n + M)
    part = torch.randn(max(slices, 1), M, n, generator=g, device=gpu_device)
    resid = torch.randn(M, n, generator=g, device=gpu_device).to(torch.bfloat16)
    gamma = (1 + 0.1 * torch.randn(n, generator=g, device=gpu_device)).to(torch.bfloat16)
    h = torch.zeros_like(resid)
    out = torch.zeros(-(-M // 32) * 32 * n, device=gpu_device, dtype=torch.bfloat16)
    L.tfd_panel_add_norm(part.data_ptr(), slices, resid.data_ptr(), h.data_ptr(),
                         gamma.data_ptr(), out.data_ptr(), M, n, 1e-6,
                         torch.cuda.current_stream().cuda_stream)
    want = resid
    if slices:
        y = part[0].clone()
        for sl in range(1, slices):
            y += part[sl]
        want = (resid.float() + y.to(torch.bfloat16).float()).to(torch.bfloat16)
    assert torch.equal(h, want)
    f = want.float()
    r = torch.rsqrt(f.pow(2).mean(-1, keepdim=True) + 1e-6)
    norm = (f * r).to(torch.bfloat16).float() * gamma.float()
    assert ((unpanel(out, M, n).float() - norm).abs() <= 2.0 ** -7 * norm.abs() + 1e-6).all()


@pytest.mark.gpu
@pytest.mark.parametrize("D,G", [(128, 2), (64, 2), (128, 1)])
@pytest.mark.parametrize("segs", [[(0, 1)], [(0, 64), (63, 1)], [(0, 200), (70, 129), (128, 3)],
                                  [(2900, 301), (0, 700)]])
def test_panel_attn(gpu_device, D, G, segs):
    """(first position, rows) segments over filled pages against f32 softmax.  Scores
    are rounded to bf16 (|s| < 8 here: 2^-6 absolute), probabilities twice and the
    output three times at 2^-9: 3e-2 of the largest |value| bounds every output."""
    L = _lib.lib()
    HKV = 2
    heads = HKV * G
    g = torch.Generator(device=gpu_device).manual_seed(D + len(segs))
    pages = -(-max(p + n for p, n in segs) // 16) + 1
    B = len(segs)
    table = torch.randperm(B * pages, generator=torch.Generator().manual_seed(1)).view(
        B, pages).to(torch.int32).to(gpu_device)
    bf = torch.bfloat16
    k = torch.randn(B * pages, HKV, 16, D, generator=g, device=gpu_device).to(bf)
    v = torch.randn(B * pages, HKV, 16, D, generator=g, device=gpu_device).to(bf)
    for b, (p0, n) in enumerate(segs):      # what lies past a context is not read
        at = torch.arange(p0 + n, pages * 16, device=gpu_device)
        rows = table[b].long()[at // 16]
        k[rows, :, at % 16] = float("nan")
        v[rows, :, at % 16] = float("nan")
        table[b, -(-(p0 + n) // 16):] = -1  # nor are the pages past it
    M = sum(n for _, n in segs)
    q = (torch.randn(M, heads, D, generator=g, device=gpu_device) * D ** -0.5).to(bf)
    qt = L.tfd_panel_attn_rows(G)
    tiles, row = [], 0
    for b, (p0, n) in enumerate(segs):
        tiles += [(row + t, min(qt, n - t), b, p0 + t) for t in range(0, n, qt)]
        row += n
    td = torch.tensor(tiles, dtype=torch.int32, device=gpu_device)
    out = torch.zeros(-(-M // 32) * 32 * heads * D, device=gpu_device, dtype=bf)
    err = torch.zeros(1, device=gpu_device, dtype=torch.int32)
    L.tfd_panel_attn(q.data_ptr(), td.data_ptr(), len(tiles), heads, HKV, D, table.data_ptr(),
                     pages, k.data_ptr(), v.data_ptr(), B * pages, out.data_ptr(),
                     err.data_ptr(), torch.cuda.current_stream().cuda_stream)
    got = unpanel(out, M, heads * D).float().view(M, heads, D)
    assert int(err.item()) == 0
    row = 0
    for b, (p0, n) in enumerate(segs):
        p = torch.arange(p0 + n, device=gpu_device)
        kc, vc = (t[table[b].long()[p // 16], :, p % 16].float().repeat_interleave(G, 1)
                  for t in (k, v))
        s = torch.einsum("mhd,phd->hmp", q[row:row + n].float(), kc)
        late = p[None, :] > (p0 + torch.arange(n, device=gpu_device))[:, None]
        a = torch.softmax(s.masked_fill(late, float("-inf")), -1)
        want = torch.einsum("hmp,phd->mhd", a, vc)
        assert (got[row:row + n] - want).abs().max() <= 3e-2 * want.abs().max()
        row += n


def _attend(device, kind, poison=None):
    """100 positions of one sequence through a prompt pass's attention -> [100][heads][D];
    *poison* sets values of ([100][KV heads][D] keys, values) before the pass reads them."""
    L = _lib.lib()
    s = torch.cuda.current_stream().cuda_stream
    n, bf, f32 = 100, torch.bfloat16, torch.float32
    D, G, HKV = {"granite": (128, 4, 2), "f32": (256, 8, 1)}.get(kind) or (*kind, 2)
    heads, pages = HKV * G, 7
    g = torch.Generator(device=device).manual_seed(D + G)
    rn = lambda *shape: torch.randn(*shape, generator=g, device=device)
    z = lambda *shape, dtype=bf: torch.zeros(*shape, device=device, dtype=dtype)
    q, k, v = rn(n, heads, D) * D ** -0.5, rn(n, HKV, D).to(bf), rn(n, HKV, D).to(bf)
    if poison is not None:
        poison(k, v)
    table = torch.tensor([5, 0, 3, 6, 1, 4, 2], dtype=torch.int32, device=device)
    kp, vp = z(pages, HKV, 16, D), z(pages, HKV, 16, D)
    at = torch.arange(n, device=device)
    qt = {"granite": _lib.PANEL_GQA_ROWS_BF16, "f32": _lib.PANEL_GQA_ROWS_F32}.get(kind) or \
        L.tfd_panel_attn_rows(G)
    tiles = torch.tensor([(t, min(qt, n - t), 0, t) for t in range(0, n, qt)],
                         dtype=torch.int32, device=device)
    out, err = z(128 * heads * D), z(1, dtype=torch.int32)
    if kind not in ("granite", "f32"):
        kp[table[at // 16].long(), :, at % 16] = k
        vp[table[at // 16].long(), :, at % 16] = v
        q = q.to(bf)
        L.tfd_panel_attn(q.data_ptr(), tiles.data_ptr(), len(tiles), heads, HKV, D,
                         table.data_ptr(), pages, kp.data_ptr(), vp.data_ptr(), pages,
                         out.data_ptr(), err.data_ptr(), s)
    else:
        if kind == "f32":                   # (query, output gate) pairs
            q = torch.stack((q, rn(n, heads, D)), 2)
        proj = torch.cat((q.reshape(n, -1).to(bf), k.reshape(n, -1), v.reshape(n, -1)), 1)
        pos, seq = at.to(torch.int32), z(n, dtype=torch.int32)
        gam, cos, sin = z(D) + 1, z(112, 64) + 1, z(112, 64)
        qw, gate, self_s = z(n * heads * D, dtype=f32), z(n * heads * D), z(n * heads, dtype=f32)
        a = _lib.TfdPanelGqaArgs()
        a.proj, a.ldp, a.M, a.err = proj.data_ptr(), proj.shape[1], n, err.data_ptr()
        a.gamma_q, a.gamma_k = gam.data_ptr(), gam.data_ptr()
        a.cos_table, a.sin_table, a.rope_rows, a.rot_dim = cos.data_ptr(), sin.data_ptr(), 112, 64
        a.pos, a.seq, a.tiles, a.ntiles = pos.data_ptr(), seq.data_ptr(), tiles.data_ptr(), \
            len(tiles)
        a.page_table, a.max_pages, a.num_pages = table.data_ptr(), pages, pages
        a.k_pool, a.v_pool, a.q, a.gate = kp.data_ptr(), vp.data_ptr(), qw.data_ptr(), \
            gate.data_ptr()
        a.self_scores, a.out, a.heads, a.kv_heads, a.head_dim = self_s.data_ptr(), \
            out.data_ptr(), heads, HKV, D
        a.scale, a.eps = (D ** -0.5, 1e-6) if kind == "f32" else (1.0, 1e-6)
        a.policy = _lib.POLICY_F32 if kind == "f32" else _lib.POLICY_BF16
        L.tfd_panel_gqa(ctypes.addressof(a), s)
    torch.cuda.synchronize()
    assert int(err.item()) == 0
    return unpanel(out, n, heads * D).float().view(n, heads, D)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [(128, 2), (64, 2), (128, 1), "granite", "f32"], ids=str)
@pytest.mark.parametrize("at", [0, 40, 70, 99])
def test_panel_attn_rows_do_not_see_what_follows_them(gpu_device, kind, at):
    """An infinite value, or a NaN key, at position *at*: the rows before it are what
    they are without it, the rows from it on take it as a step takes it (an infinity of
    that dimension alone; NaN throughout).  Rows taken position by position differ from
    the tiles' by f32 orders, whose roundings test_panel_attn bounds: 3e-2 of the
    largest value."""
    clean = _attend(gpu_device, kind)
    bar = 3e-2 * clean.abs().max()
    rows = torch.arange(100, device=gpu_device)

    def infinite(k, v):
        v[at, 0, 5] = float("inf")

    def nan_key(k, v):
        k[at, 0] = float("nan")

    mine = slice(0, clean.shape[1] // (1 if kind == "f32" else 2))   # kv head 0's query heads
    got = _attend(gpu_device, kind, infinite)
    seen = torch.zeros_like(clean, dtype=torch.bool)
    seen[at:, mine, 5] = True
    assert got[seen].isinf().all()
    assert ((got - clean).abs()[~seen] <= bar).all()
    got = _attend(gpu_device, kind, nan_key)
    assert got[rows >= at][:, mine].isnan().all()
    seen = torch.zeros_like(clean, dtype=torch.bool)
    seen[at:, mine] = True
    assert ((got - clean).abs()[~seen] <= bar).all()


@pytest.mark.gpu
def test_panel_attn_probabilities_are_exactly_rounded(gpu_device):
    """p = bf16(exp(x)) for every bf16 x in (-87, 0] (its result a normal number): one
    sequence per x, a past key that scores x beside the row's own, which scores 0.  The
    output p * 1 / bf16(p + 1), taken in f32 and rounded, is equal to the bit."""
    L = _lib.lib()
    x = torch.arange(0x8000, 0xc2ae, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    n, D, bf = len(x), 64, torch.bfloat16
    z = lambda *shape, dtype=bf: torch.zeros(*shape, device=gpu_device, dtype=dtype)
    q, k, v = z(n, 2, D), z(n, 1, 16, D), z(n, 1, 16, D)
    q[:, :, 0], k[:, 0, 0, 0], v[:, 0, 0, 0] = 1, x.to(gpu_device), 1
    i = torch.arange(n, dtype=torch.int32, device=gpu_device)
    tiles = torch.stack((i, torch.ones_like(i), i, torch.ones_like(i)), 1).contiguous()
    out, err = z(-(-n // 32) * 32 * 2 * D), z(1, dtype=torch.int32)
    L.tfd_panel_attn(q.data_ptr(), tiles.data_ptr(), n, 2, 1, D, i.data_ptr(), 1, k.data_ptr(),
                     v.data_ptr(), n, out.data_ptr(), err.data_ptr(),
                     torch.cuda.current_stream().cuda_stream)
    got = unpanel(out, n, 2 * D).view(n, 2, D)[:, :, 0].cpu()
    assert int(err.item()) == 0
    p = torch.exp(x.double()).to(bf).float()
    want = (p * (1 / (p + 1).to(bf).float())).to(bf)
    off = (got != want[:, None]).sum()
    assert off == 0, (int(off), x[(got != want[:, None]).any(1)][:8].tolist())


@pytest.mark.gpu
def test_passes_cut_anywhere_fill_the_same_cache(gpu_device, monkeypatch):
    """Three prompts in one pass and in passes of 64 rows: the same caches to the
    bf16 bar (other GEMM shapes, other f32 orders)."""
    from tests._parity import assert_close_bf16
    from tests.test_gpu_engine import SMALL, _prompt
    from tilefoundry_amd.qwen3 import prefill, synthetic_weights
    from tilefoundry_amd.qwen3.batch_engine import BatchEngine

    w = synthetic_weights(SMALL, seed=1, norms="ones")
    prompts = [_prompt(n, SMALL.vocab_size, seed=n) for n in (90, 2, 71)]
    eng = BatchEngine(SMALL, w, batch=3, device=gpu_device, max_new=8, prompt_room=96)
    eng.kpool.zero_()                       # the capture's own steps left rows behind
    eng.vpool.zero_()
    eng.prefill(prompts)
    k, v = eng.kpool.clone(), eng.vpool.clone()
    monkeypatch.setattr(prefill, "MAX_PASS", 64)
    eng.kpool.zero_()
    eng.vpool.zero_()
    eng.prefill(prompts)
    eng.check_errors()
    assert_close_bf16(eng.kpool, k, max_rel=2e-2, name="k")
    assert_close_bf16(eng.vpool, v, max_rel=2e-2, name="v")


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
def test_panel_moe_with_uneven_picks(gpu_device, fp8):
    """Experts picked by none, 1, 63, 64, 65 and 207 of 200 rows (two slots each): every
    entry's two projections against f64 sums.  hidden is rounded twice more before its
    own rounding (gate, up; 2^-9 each), the output once: 2^-6 of the output's norm."""
    L = _lib.lib()
    s = torch.cuda.current_stream().cuda_stream
    M, k, E, H, I = 200, 2, 7, 512, 256
    g = torch.Generator(device=gpu_device).manual_seed(5 + fp8)
    counts = [0, 1, 63, 64, 65, 207, 0]
    picks = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    idx = picks[torch.randperm(M * k, generator=torch.Generator().manual_seed(2))].view(M, k)
    rn = lambda *shape: torch.randn(*shape, generator=g, device=gpu_device)
    x = rn(M, H).to(torch.bfloat16)
    a = _lib.TfdPanelMoeArgs()
    keep, mats = [], {}
    for name, rows, cols in (("gate", I, H), ("up", I, H), ("down", H, I)):
        w = rn(E * rows, cols)
        if fp8:
            w8 = w.to(torch.float8_e4m3fn)
            sc = torch.rand(E * rows, generator=g, device=gpu_device) * 0.05 + 0.05
            packed = torch.empty(E * rows * cols, dtype=torch.uint8, device=gpu_device)
            L.tfd_pack_skinny_fp8(w8.data_ptr(), cols, E * rows, cols, packed.data_ptr(), s)
            keep += [w8, sc, packed]
            setattr(a, f"w_{name}", packed.data_ptr())
            setattr(a, f"s_{name}", sc.data_ptr())
            mats[name] = (w8.double() * sc.double()[:, None]).view(E, rows, cols)
        else:
            w = (0.08 * w).to(torch.bfloat16)
            keep.append(w)
            setattr(a, f"w_{name}", w.data_ptr())
            mats[name] = w.double().view(E, rows, cols)
    z = lambda n, dtype=torch.bfloat16: torch.zeros(n, dtype=dtype, device=gpu_device)
    idxd = idx.to(torch.int32).to(gpu_device)
    hidden, d, err = z(M * k * I), z(M * k * H), z(1, torch.int32)
    groups = z(_lib.panel_moe_words(E, M * k), torch.int32)
    a.x, a.idx, a.groups, a.hidden, a.d = (t.data_ptr() for t in (x, idxd, groups, hidden, d))
    a.M, a.k, a.experts, a.H, a.I, a.fp8 = M, k, E, H, I, int(fp8)
    a.policy, a.err = _lib.POLICY_BF16 if fp8 else _lib.POLICY_F32, err.data_ptr()
    L.tfd_panel_moe(ctypes.addressof(a), s)
    got = d.view(M, k, H).double()
    assert int(err.item()) == 0
    xd = x.double()
    for m in range(M):
        for j in range(k):
            e = int(idx[m, j])
            h = torch.nn.functional.silu(mats["gate"][e] @ xd[m]) * (mats["up"][e] @ xd[m])
            want = mats["down"][e] @ h
            assert (got[m, j] - want).norm() <= 2.0 ** -6 * want.norm(), (m, j, e)


def test_token_array_takes_what_a_prompt_may_be():
    """Lists, tuples, arrays and tensors of ids; what does not fit is refused."""
    import numpy as np

    from tilefoundry_amd.qwen3.prefill import in_vocab, int32_ids, token_array

    for p in ([1, 2, 3], (1, 2, 3), np.array([1, 2, 3], np.int32), torch.tensor([1, 2, 3]),
              [torch.tensor(1), 2, np.int64(3)]):
        assert token_array(p).tolist() == [1, 2, 3] and token_array(p).dtype == np.int64
    assert token_array([]).size == 0 and in_vocab(token_array([]), 5)
    assert in_vocab(token_array([0, 4]), 5)
    assert not in_vocab(token_array([0, 5]), 5) and not in_vocab(token_array([-1]), 5)
    with pytest.raises(ValueError):
        token_array([1 << 70])
    with pytest.raises(ValueError):
        token_array([[1, 2], [3, 4]])
    with pytest.raises(RuntimeError):
        int32_ids([(1 << 32) + 5])


def test_token_array_takes_tensors_of_one_element():
    """Ids as a sampling loop leaves them; text, rows and NaN are refused."""
    import numpy as np

    from tilefoundry_amd.qwen3.prefill import token_array

    for p in ([torch.tensor([1]), torch.tensor([2])], [torch.tensor([1]), 2],
              (torch.tensor([[1]]), torch.tensor(2)), torch.tensor([1, 2], dtype=torch.int32),
              [1.0, 2.5], torch.tensor([1.0, 2.0]), [torch.tensor([1.5]), 2], np.array([1.0, 2.0])):
        assert token_array(p).tolist() == [1, 2] and token_array(p).dtype == np.int64
    for p in ("12", ["1", "2"], torch.tensor([[1], [2]]), np.array([[1], [2]]), [[1], [2]], 3,
              [None], [torch.tensor([1, 2]), 3], [float("nan")], np.array([np.inf])):
        with pytest.raises((ValueError, RuntimeError)):
            token_array(p)


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [8, 9, 17, 32])
def test_batch_step_on_both_sides_of_nine_rows(gpu_device, batch):
    """From nine rows on a step's o and down (from 17, gate/up) projections are panel GEMMs
    with the norm behind them: the first, middle and last sequence against the
    oracle, as the smaller batches are checked."""
    from tests.test_gpu_batch import _oracle_runs
    from tests.test_gpu_engine import SMALL, _check_run, _prompt
    from tilefoundry_amd.qwen3 import synthetic_weights
    from tilefoundry_amd.qwen3.batch_engine import BatchEngine

    w = synthetic_weights(SMALL, seed=2, norms="ones")
    prompts = [_prompt(3 + b % 5, SMALL.vocab_size, seed=b) for b in range(batch)]
    eng = BatchEngine(SMALL, w, batch=batch, device=gpu_device, max_new=12, prompt_room=8)
    run = eng.generate(prompts, 12, record_logits=True)
    some = [0, batch // 2, batch - 1]
    for b, orc in zip(some, _oracle_runs(SMALL, w, [prompts[b] for b in some], 12)):
        seq = type("Run", (), {"tokens": run.tokens[b], "logits": run.logits[b]})
        _check_run(seq, orc, 12, strict=False)
