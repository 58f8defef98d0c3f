"""GPU parity of the fused DiT glue (bd3_ln_modulate, bd3_gate_residual,
bd3_gate_residual_ln_modulate) against oracle/dit.py: the gated residual
bit-exact in every dtype mix; the residual + LayerNorm fusion bit-exact with
the two calls it replaces;
LayerNorm + modulate within the rounding its fp32 row statistics allow
(summation order differs): fp32 results within 1e-5 relative, bf16 results
within one bf16 ulp per rounding of the magnitudes entering the last add, at most 1% of
elements off by any amount."""
from __future__ import annotations

import pytest
import torch

from kernels.dit_glue import gate_residual, ln_modulate
from oracle.dit import gate_residual as ref_gate
from oracle.dit import layer_norm as ref_layer_norm
from oracle.dit import ln_modulate as ref_lnmod

F32, BF = torch.float32, torch.bfloat16


def rnd(shape, dtype, seed, scale=1.0, shift=0.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale + shift).to(dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("xd,md,od", [(F32, BF, F32), (F32, BF, BF), (BF, BF, BF), (BF, F32, F32), (F32, F32, F32)])
# One row a wave (two waves a row at d = 4096; several rows a wave: below); d =
# 520 leaves two lanes with a third, last chunk.
@pytest.mark.parametrize("B,S,D", [(2, 37, 768), (1, 5, 64), (8, 256, 768), (2, 9, 2048), (3, 7, 4096),
                                   (2, 11, 520)])
def test_ln_modulate(cuda, xd, md, od, B, S, D):
    print(f"ln_modulate x={xd} mod={md} out={od} shape=({B},{S},{D})", flush=True)
    x = rnd((B, S, D), xd, 1, scale=2.0, shift=0.3)
    w = rnd((D,), F32, 2, scale=0.2, shift=1.0)
    sh, sc = rnd((B, D), md, 3, 0.5), rnd((B, D), md, 4, 0.5)
    want = ref_lnmod(x, w, sh, sc)
    got = ln_modulate(x.to(cuda), w.to(cuda), sh.to(cuda)[:, None], sc.to(cuda)[:, None],
                      out_dtype=od if od != want.dtype else None).cpu()
    assert got.dtype == od
    if od == F32 and xd == F32:
        assert torch.allclose(got, want.float(), rtol=1e-5, atol=1e-5)
    else:
        # A row statistic one fp32 ulp off can move a rounding to bf16 (of y
        # when x is bf16, then of the product and of the sum on the bf16
        # path) by one bf16 ulp each, i.e. at most 2^-7 relative per rounding:
        # within 3 * 2^-7 of the magnitudes entering the last add.
        h = ref_layer_norm(x, w).float()
        mag = (h * (1 + sc.float()[:, None])).abs() + sh.float()[:, None].abs()
        diff = (got.float() - want.to(od).float()).abs()
        assert (diff <= 3 * 2.0 ** -7 * mag + 1e-30).all(), float((diff / (mag + 1e-30)).max())
        assert (diff > 0).float().mean() < 0.01, float((diff > 0).float().mean())


@pytest.mark.gpu
@pytest.mark.parametrize("xd,gd,yd", [(F32, BF, BF), (BF, BF, BF), (F32, F32, F32), (BF, F32, BF)])
@pytest.mark.parametrize("B,S,D", [(3, 50, 768), (2, 7, 520), (1, 3, 64)])
def test_gate_residual_bit_exact(cuda, xd, gd, yd, B, S, D):
    x, g, y = rnd((B, S, D), xd, 5), rnd((B, D), gd, 6), rnd((B, S, D), yd, 7)
    want = ref_gate(x, g, y)
    got = gate_residual(x.to(cuda), g.to(cuda)[:, None], y.to(cuda)).cpu()
    assert got.dtype == want.dtype and torch.equal(got, want)


@pytest.mark.gpu
def test_gate_residual_in_place(cuda):
    x = rnd((2, 16, 64), F32, 8).to(cuda)
    g, y = rnd((2, 64), BF, 9).to(cuda), rnd((2, 16, 64), BF, 10).to(cuda)
    want = ref_gate(x.cpu(), g.cpu(), y.cpu())
    out = gate_residual(x, g, y, out=x)
    assert out.data_ptr() == x.data_ptr() and torch.equal(x.cpu(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("xd,md,yd,od", [(BF, BF, BF, BF), (F32, BF, BF, None), (F32, BF, BF, BF),
                                         (BF, F32, BF, None), (F32, F32, F32, None)])
@pytest.mark.parametrize("B,S,D", [(2, 37, 768), (1, 5, 64), (3, 2, 4096), (2, 9, 2048), (2, 11, 520)])
def test_gate_residual_ln_modulate_matches_two_calls(cuda, xd, md, yd, od, B, S, D):
    """The fused residual + LayerNorm + modulate equals gate_residual followed
    by ln_modulate bit for bit (same kernels' arithmetic, one launch), both
    outputs, including the in-place residual update; vectors sliced from one
    (batch, 6, 1, d) adaLN tensor as the model does."""
    from kernels.dit_glue import gate_residual_ln_modulate
    print(f"gate_residual_ln_modulate x={xd} mod={md} y={yd} out={od} shape=({B},{S},{D})", flush=True)
    x = rnd((B, S, D), xd, 11, scale=2.0, shift=0.3).to(cuda)
    y = rnd((B, S, D), yd, 12).to(cuda)
    ada = rnd((B, 6, 1, D), md, 13, 0.5).to(cuda)
    g, sh, sc = ada[:, 2], ada[:, 3], ada[:, 4]
    w = rnd((D,), F32, 14, scale=0.2, shift=1.0).to(cuda)
    want_x = gate_residual(x, g, y)
    want_h = ln_modulate(want_x, w, sh, sc, out_dtype=od)
    got_x, got_h = gate_residual_ln_modulate(x, g, y, w, sh, sc, out_dtype=od)
    assert got_x.dtype == want_x.dtype and got_h.dtype == want_h.dtype
    assert torch.equal(got_x, want_x) and torch.equal(got_h, want_h)
    if got_x.dtype == x.dtype:  # in place
        x2 = x.clone()
        got_x2, got_h2 = gate_residual_ln_modulate(x2, g, y, w, sh, sc, out_dtype=od, x_out=x2)
        assert got_x2.data_ptr() == x2.data_ptr()
        assert torch.equal(x2, want_x) and torch.equal(got_h2, want_h)
    # gate and the modulation vectors from different adaLN tensors (the last
    # layer's gate with the final layer's shift / scale): batch strides differ
    fin = rnd((B, 2, 1, D), md, 15, 0.5).to(cuda)
    want_h3 = ln_modulate(want_x, w, fin[:, 0], fin[:, 1], out_dtype=od)
    _, got_h3 = gate_residual_ln_modulate(x, g, y, w, fin[:, 0], fin[:, 1], out_dtype=od)
    assert torch.equal(got_h3, want_h3)


@pytest.mark.gpu
@pytest.mark.parametrize("xd", [F32, BF])
# 16383 rows: one per wave; 16384 and 24579: two and three, an odd sequence
# length, so a wave's rows lie in two batch entries; 65537: eight, and a last
# wave with one. d = 64, 264, 768, 1016: one to four chunks a lane, the last
# chunk of 264 and 1016 not in every lane.
@pytest.mark.parametrize("B,S,D", [(3, 5461, 768), (4, 4096, 264), (3, 8193, 1016), (65537, 1, 64)])
def test_several_rows_per_wave(cuda, xd, B, S, D):
    from kernels.dit_glue import gate_residual_ln_modulate
    print(f"rows per wave x={xd} shape=({B},{S},{D})", flush=True)
    g = torch.Generator(device=cuda).manual_seed(21)
    x, y = (torch.randn(B, S, D, generator=g, device=cuda) for _ in range(2))
    x, y = (2 * x + 0.3).to(xd), y.to(BF)
    ada = (0.5 * torch.randn(B, 6, 1, D, generator=g, device=cuda)).to(BF)
    gate, sh, sc = ada[:, 2], ada[:, 3], ada[:, 4]
    w = 1 + 0.2 * torch.randn(D, generator=g, device=cuda)
    want_x = ref_gate(x, gate[:, 0], y)
    got_x, got_h = gate_residual_ln_modulate(x, gate, y, w, sh, sc, out_dtype=BF)
    assert torch.equal(got_x, want_x)
    assert torch.equal(got_h, ln_modulate(want_x, w, sh, sc, out_dtype=BF))
    # test_ln_modulate's bound: one bf16 ulp per rounding of the magnitudes entering the last add
    h = ref_layer_norm(want_x, w).float()
    want = (h.to(xd) * (1 + sc) + sh).to(BF).float()
    mag = (h * (1 + sc.float())).abs() + sh.float().abs()
    diff = (got_h.float() - want).abs()
    assert (diff <= 3 * 2.0 ** -7 * mag + 1e-30).all(), float((diff / (mag + 1e-30)).max())
    assert (diff > 0).float().mean() < 0.01, float((diff > 0).float().mean())


@pytest.mark.gpu
# Two waves to a row. 2056: one lane of the first wave with a fifth chunk and
# none of the second; 2304: half of the first wave; 3072: six chunks a lane;
# 3080, 4088: a seventh, an eighth not in every lane.
@pytest.mark.parametrize("D", [2056, 2304, 3072, 3080, 4088])
def test_rows_of_two_waves(cuda, D):
    for xd, md, od in ((F32, BF, F32), (F32, BF, BF), (BF, BF, BF), (BF, F32, F32), (F32, F32, F32)):
        test_ln_modulate(cuda, xd, md, od, 3, 5, D)
    for xd, md, yd, od in ((BF, BF, BF, BF), (F32, BF, BF, None), (BF, F32, BF, None), (F32, F32, F32, None),
                           (BF, BF, F32, None), (BF, F32, F32, None), (F32, BF, F32, None), (F32, F32, BF, None)):
        test_gate_residual_ln_modulate_matches_two_calls(cuda, xd, md, yd, od, 3, 5, D)


@pytest.mark.gpu
# 2^24 + 4096 rows of 1032 and of 2056 (two launches; one and two waves a row), 2^29
# + 8192 of 8 (17 rows a wave; waves * 64 does not fit 32 bits).
@pytest.mark.parametrize("B,S,D", [(4097, 4096, 1032), (4097, 4096, 2056), (131074, 4096, 8)])
def test_very_many_rows(cuda, B, S, D):
    """One sequence repeated by a batch stride of 0: every entry of the
    result is the first one's, which a call of one sequence gives."""
    print(f"rows {B} x {S} x {D}", flush=True)
    x, w, m = rnd((1, S, D), BF, 31).to(cuda), rnd((D,), F32, 32).to(cuda), rnd((1, D), BF, 33).to(cuda)
    want = ln_modulate(x, w, m, m)
    got = ln_modulate(x.expand(B, S, D), w, m.expand(B, D), m.expand(B, D))
    for b in range(0, B, 256):
        assert torch.equal(got[b:b + 256], want.expand(min(256, B - b), S, D)), b
