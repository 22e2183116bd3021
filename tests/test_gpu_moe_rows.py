"""fp8 experts for more than 16 rows (the matrix-core kernels over row-major
weights in csrc/hybrid.hip) against the oracle: one row past the packed limit, an
expert picked by more rows than a pass holds, every column remainder, and widths
that keep the lane-wise kernels."""
import pytest
import torch

from oracle import hybrid_ref as H
from tests._parity import assert_close_bf16
from tests.test_gpu_hybrid import BF, _fp8_codes, _moe_call, _routing
from tilefoundry_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,same,hs,inter,sh,E,k", [
    (17, False, 512, 128, 256, 12, 4),
    (32, True, 256, 384, 128, 6, 2),        # 384 columns: whole blocks; all rows on two experts
    (40, True, 384, 128, 128, 8, 3),        # more entries than a pass holds; 384 = 3 x 128
    (32, False, 4096, 768, 1536, 16, 10),   # Granite's widths
    (20, False, 448, 192, 64, 12, 4),       # not whole pieces: the lane-wise kernels
])
def test_fp8_experts_past_sixteen_rows(gpu_device, rows, same, hs, inter, sh, E, k):
    """The bar of the lane-wise kernels' own test: one bf16 rounding per step, f32
    sums in another order."""
    g = torch.Generator().manual_seed(rows + hs)
    x = H.bf(torch.randn(rows, hs, generator=g))
    weights, idx = _routing(rows, E, k, g)
    if same:
        idx = idx[:1].repeat(rows, 1)
    weights = H.bf(weights)
    sc = lambda *s: torch.rand(*s, generator=g) * 0.004 + 0.002
    gc, uc, dc = _fp8_codes((E, inter, hs), g), _fp8_codes((E, inter, hs), g), \
        _fp8_codes((E, hs, inter), g)
    gs, us, ds = sc(E, inter), sc(E, inter), sc(E, hs)
    sic, soc = _fp8_codes((2 * sh, hs), g), _fp8_codes((hs, sh), g)
    sis, sos = sc(2 * sh), sc(hs)
    got = _moe_call(x, weights, idx, w_gate=gc, w_up=uc, w_down=dc, w_sin=sic, w_sout=soc,
                    s=(gs, us, ds, sis, sos), fp8=True, policy=_lib.POLICY_BF16)
    want = H.moe_c5(x, weights, idx, gc, gs, uc, us, dc, ds, sic, sis, soc, sos)
    assert torch.equal(got, got.to(BF).float())
    assert_close_bf16(got, want, max_rel=2e-2, min_cos=0.9999, name="moe rows")
