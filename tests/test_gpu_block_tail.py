"""GPU checks of the one-launch block tail (out-projection, LN2, feed-forward, next norm at
width 128) where its 32-row blocks and the workgroups' shares of them end.

Reference: float64 torch on the same 16-bit operands, unrounded between the products.  The
tolerance follows the two fp16 intermediates through: a relative 2^-11 on every h2 gives at
most `2^-11 |h2| |W1|^T` on the hidden sums, times GELU's largest slope 1.13 and with f's own
2^-11 gives `df`, `df |W2|^T` on r2, and LayerNorm's derivative that on the output, plus the
output's own rounding; 2^-17 of the row's largest value covers the fp32 sums.
"""

import pytest
import torch

from _gpu_util import DEV

pytestmark = pytest.mark.gpu
D = 128
EPS = 1e-5


def _operands(M, resid_dtype, seed):
    g = torch.Generator().manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=g)
    w = [(rn(D, D) * D ** -0.5).half().to(DEV) for _ in range(3)]
    par = [(rn(D) + (1.0 if i in (1, 5) else 0.0)).to(DEV) for i in range(7)]  # bo g2 b2n b1 b2 gn bn
    return rn(M, D).half().to(DEV), (rn(M, D) * 2 + 1).to(resid_dtype).to(DEV), w, par


def _tail(ctx, resid, w, p, **kw):
    from cobra_amd import ops

    return ops.block_tail(ctx, resid, w[0], p[0], p[1], p[2], w[1], p[3], w[2], p[4], p[5], p[6], eps=EPS, **kw)


def _ln(r, gm, bt):
    mean = r.mean(1, keepdim=True)
    rstd = ((r - mean).square().mean(1, keepdim=True) + EPS).rsqrt()
    xh = (r - mean) * rstd
    return xh * gm + bt, xh, rstd


def _reference(ctx, resid, w, par, rm, mask_out):
    wd, p = [x.double() for x in w], [x.double() for x in par]
    mv = torch.ones(ctx.shape[0], 1, device=DEV, dtype=torch.float64) if rm is None else rm.double()[:, None]
    r1 = resid.double() + (ctx.double() @ wd[0].t() + p[0]) * mv
    h2, _, _ = _ln(r1, p[1], p[2])
    f = torch.nn.functional.gelu(h2 @ wd[1].t() + p[3])
    r2 = (r1 + f @ wd[2].t() + p[4]) * mv
    out, xh, rstd = _ln(r2, p[5], p[6])
    u = 2.0 ** -11
    df = u * f.abs() + 1.13 * u * (h2.abs() @ wd[1].abs().t())
    dr = (df @ wd[2].abs().t()) * mv + 2.0 ** -17 * r1.abs().amax(1, keepdim=True)
    dx = rstd * (dr + dr.mean(1, keepdim=True) + xh.abs() * (xh.abs() * dr).mean(1, keepdim=True))
    if mask_out:
        out = out * mv
    return r2, dr, out, dx * p[5].abs() + 1e-6


def _check(M, resid_dtype, masked, last, fp16_out, in_place=False):
    ctx, resid, w, par = _operands(M, resid_dtype, 7 * M + masked)
    rm = (torch.rand(M, generator=torch.Generator().manual_seed(M)) < 0.6).to(DEV) if masked else None
    r2, dr, want, dy = _reference(ctx, resid, w, par, rm, last and masked)
    r_out = None if last else (resid if in_place else torch.full((M, D), float("nan"), device=DEV))
    got = _tail(ctx, resid, w, par, rmask=rm, r_out=r_out, norm_fp16=fp16_out, mask_out=last)
    what = (M, resid_dtype, masked, last, fp16_out, in_place)
    dy = dy + (2.0 ** -11 * want.abs() if fp16_out else 0.0)
    assert got.dtype == (torch.float16 if fp16_out else torch.float32)
    assert bool(((got.double() - want).abs() <= dy).all()), what
    if r_out is not None:
        assert bool(((r_out.double() - r2).abs() <= dr).all()), what


@pytest.mark.parametrize("M", [1, 2, 31, 32, 33, 63, 64, 65, 96, 127, 1000, 16383, 16384, 16385, 24577, 49153, 65536,
                               100003])
def test_block_ends(M):
    for masked in (False, True):
        _check(M, torch.float16, masked, False, True)
        _check(M, torch.float32, masked, False, True)
        _check(M, torch.float32, masked, False, True, in_place=True)
        _check(M, torch.float32, masked, True, True)
        _check(M, torch.float32, masked, True, False)
        _check(M, torch.float16, masked, True, False)
    print(f"[block-tail] M={M} ok", flush=True)


def test_rows_keep_to_themselves_and_repeat():
    """Rows that are not finite stay alone in their block, and a second run gives the same bits."""
    ctx, resid, w, par = _operands(4099, torch.float32, 5)
    clean = _tail(ctx, resid, w, par)
    assert torch.equal(clean, _tail(ctx, resid, w, par))
    ctx[70] = float("inf")
    resid[4098] = float("nan")
    got = _tail(ctx, resid, w, par)
    keep = torch.ones(4099, dtype=torch.bool, device=DEV)
    keep[70] = keep[4098] = False
    assert torch.equal(got[keep], clean[keep]) and not torch.isfinite(got[~keep]).any()
    # a masked row's branch is dropped, infinite or not, and an all-constant row has no variance
    rm = torch.ones(4099, dtype=torch.bool, device=DEV)
    rm[70] = False
    resid[4098] = 3.0
    masked = _tail(ctx, resid, w, par, rmask=rm, mask_out=True)
    assert torch.isfinite(masked).all() and bool((masked[70] == 0).all())


def test_arguments():
    from cobra_amd import CobraError, ops

    ctx, resid, w, par = _operands(64, torch.float32, 3)
    with pytest.raises(CobraError):  # an fp32 output and a residual share their place on chip
        _tail(ctx, resid, w, par, r_out=torch.empty_like(resid), norm_fp16=False)
    both = torch.empty(96, D, device=DEV)
    with pytest.raises(CobraError):  # r_out over another row's residual
        _tail(ctx, both[:64], w, par, r_out=both[32:])
    with pytest.raises(ValueError):
        _tail(ctx[:, :64].contiguous(), resid, w, par)
    with pytest.raises(ValueError):
        _tail(ctx, resid[:32], w, par)
    # biases and norm parameters may be views at any element of a larger buffer
    views = [torch.cat([p.new_zeros(1 + i % 3), p])[1 + i % 3:] for i, p in enumerate(par)]
    assert torch.equal(_tail(ctx, resid, w, views), _tail(ctx, resid, w, par))
    assert ops.block_tail_ok(128, 128) and not ops.block_tail_ok(128, 512) and not ops.block_tail_ok(256, 128)
    assert _tail(ctx[:0], resid[:0], w, par).shape == (0, D)
