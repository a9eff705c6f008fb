"""GPU checks of the causal and the key-masked attention where blocks and tiles end.

Sequence lengths on both sides of a 32-key tile, a 64-key mask word, a 128-key block and a
256-query workgroup; every head-dim class and some head dims below their class's width;
token masks that end a sequence early, start it late, leave holes, or empty it; and logits
moved far up and down, so that a wave's first tiles are refused and its references move
(an added constant per query leaves the softmax itself unchanged).

Reference: fp32 torch softmax attention on the same 16-bit values (TTB:98-113); gate of the
other attention op tests (`allclose(atol=2e-3, rtol=1e-2)`, bf16 `atol=1.6e-2, rtol=2e-2`:
the rounding of the probabilities and of the output, 2^-11 / 2^-8 of values of order 1).
"""

import math

import pytest
import torch

from _gpu_util import DEV

pytestmark = pytest.mark.gpu


def _mask(kind, B, S, g):
    j = torch.arange(S)[None, :]
    if kind == "none":
        return None
    if kind == "tail":
        return j < torch.randint(1, S + 1, (B, 1), generator=g)
    if kind == "head":
        return j >= torch.randint(0, S, (B, 1), generator=g)
    m = torch.rand(B, S, generator=g) < 0.6
    m[0] = False
    return m


def _reference(qkv, B, S, H, hd, causal, mask):
    q, k, v = qkv.float().view(B, S, 3, H, hd).permute(2, 0, 3, 1, 4)
    s = (q @ k.transpose(-2, -1).contiguous()) * hd ** -0.5
    dead = torch.zeros(B, 1, S, S, dtype=torch.bool, device=qkv.device)
    if mask is not None:
        dead = dead | ~mask[:, None, None, :]
    if causal:
        dead = dead | torch.ones(S, S, dtype=torch.bool, device=qkv.device).triu(1)
    p = torch.softmax(s.masked_fill(dead, float("-inf")), -1).nan_to_num(0.0)
    return (p @ v).transpose(1, 2).reshape(B * S, H * hd)


@pytest.mark.parametrize("hd", [8, 16, 32, 40, 64, 128, 200, 256])
@pytest.mark.parametrize("causal,kind", [(True, "none"), (False, "tail"), (True, "tail"), (True, "head"),
                                         (False, "holes"), (True, "holes")])
@pytest.mark.parametrize("offset", [0.0, 40.0, -40.0])
def test_attn_edges(hd, causal, kind, offset):
    from cobra_amd import ops

    B, H = 3, 2
    for S in (1, 31, 33, 64, 65, 127, 129, 256, 257, 333):
        g = torch.Generator().manual_seed(S * 7 + hd)
        q, k, v = torch.randn(3, B, S, H, hd, generator=g)
        if offset:
            q[..., 0], k[..., 0] = hd ** 0.5, offset  # adds `offset` to every logit
        qkv = torch.stack([q, k, v], 2).reshape(B * S, 3 * H * hd)
        mask = _mask(kind, B, S, g)
        for dt in (torch.float16, torch.bfloat16) if offset == 0.0 else (torch.float16,):
            x = qkv.to(dt).to(DEV)
            m = None if mask is None else mask.to(DEV)
            got = ops.attn(x, B, S, H, hd, hd ** -0.5, causal=causal, key_mask=m).float()
            want = _reference(x, B, S, H, hd, causal, m)
            tol = dict(atol=2e-3, rtol=1e-2) if dt == torch.float16 else dict(atol=1.6e-2, rtol=2e-2)
            err = (got - want).abs().max().item()
            assert torch.allclose(got, want, **tol), (hd, S, causal, kind, offset, dt, err)
    print(f"[attn-edges] hd{hd} causal={causal} mask={kind} offset={offset} ok", flush=True)


@pytest.mark.parametrize("hd", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_noncausal_waves_past_the_end(hd, dt):
    """Without a mask, on both sides of where a workgroup's last wave has no query, for
    workgroups of 2, 4 and 8 waves, over one key block and several (at 730 the one such wave of
    24 computes)."""
    from cobra_amd import ops

    B, H = 3, 2
    for S in (32, 33, 64, 65, 96, 97, 128, 129, 224, 225, 256, 257, 480, 481, 513, 700, 730):
        g = torch.Generator().manual_seed(S * 3 + hd)
        x = torch.randn(B * S, 3 * H * hd, generator=g).to(dt).to(DEV)
        got = ops.attn(x, B, S, H, hd, hd ** -0.5, causal=False).float()
        want = _reference(x, B, S, H, hd, False, None)
        tol = dict(atol=2e-3, rtol=1e-2) if dt == torch.float16 else dict(atol=1.6e-2, rtol=2e-2)
        assert torch.allclose(got, want, **tol), (hd, S, (got - want).abs().max().item())


@pytest.mark.parametrize("hd", [64, 256])
def test_masked_attention_repeats_bit_for_bit(hd):
    """Sharp logits and a mask ending inside a tile: references move at many places, and two
    launches agree bit for bit (each output has one owner and a fixed order of sums)."""
    from cobra_amd import ops

    B, S, H = 4, 1001, 2
    g = torch.Generator().manual_seed(hd)
    x = (torch.randn(B * S, 3 * H * hd, generator=g) * 2.0).half().to(DEV)
    mask = (torch.arange(S)[None, :] < torch.tensor([[1001], [870], [613], [40]])).to(DEV)
    got = ops.attn(x, B, S, H, hd, hd ** -0.5, causal=False, key_mask=mask)
    assert torch.equal(got, ops.attn(x, B, S, H, hd, hd ** -0.5, causal=False, key_mask=mask))
    want = _reference(x, B, S, H, hd, False, mask)
    assert torch.allclose(got.float(), want, atol=8e-3, rtol=1e-2)  # v is twice as large, p up to 1: 4x the rounding


@pytest.mark.parametrize("hd", [16, 32, 64, 128])
@pytest.mark.parametrize("masked", [False, True])
def test_causal_keys_far_below_a_low_maximum(hd, masked):
    """A row whose scores all lie below zero: 32 keys near 2^-5.9, thousands near 2^-17.

    Relative to the row's maximum the many are normal fp16 numbers, so each probability is
    rounded by 2^-11 of itself at most, and the output is off by at most
    `2^-11 sum_j w_j |v_j - out|` plus its own rounding (2^-11 |out|) and the fp32 sums (2^-18).
    Relative to 0 they would be subnormal, and the error up to 2^-8 of each."""
    from cobra_amd import ops

    B, S, H = 1, 4096, 2
    q, k, v = torch.zeros(3, B, S, H, hd)
    q[..., 0] = -5.9
    q[..., 1] = torch.linspace(-17.0, -16.0, S)[None, :, None]
    k[:, :32, :, 0] = 1.0
    k[:, 32:, :, 1] = 1.0
    v[:, 32:] = 1.0
    x = torch.stack([q, k, v], 2).reshape(B * S, 3 * H * hd).half().to(DEV)
    mask = (torch.arange(S)[None, :] < S - 3).to(DEV) if masked else None
    got = ops.attn(x, B, S, H, hd, math.log(2.0), causal=True, key_mask=mask).double()[:, 0]  # log2 units as given
    few = 32 * 2.0 ** x[:, 0].double()
    n = (torch.arange(S, device=DEV) - 31).clamp(min=0, max=S - 35 if masked else S)
    many = n * 2.0 ** x[:, 1].double()
    few[:31] = 1.0  # rows before the 32nd key: only keys with v = 0
    out = many / (few + many)
    tol = 2.0 ** -11 * (2 * out * (1 - out) + out) + 2.0 ** -18
    err = (got - out).abs()
    assert bool((err <= tol).all()), (hd, masked, (err / tol).max().item())


@pytest.mark.parametrize("B,H", [(1, 7), (2, 4), (3, 3), (13, 5), (11, 7), (100, 3)])
@pytest.mark.parametrize("masked", [False, True])
def test_causal_many_pairs(B, H, masked):
    """Every (sequence, head, query block) is computed: pair counts on both sides of 8 and
    not in whole groups of 8 per XCD, one to three query blocks."""
    from cobra_amd import ops

    hd = 32
    for S in (130, 257, 600):
        g = torch.Generator().manual_seed(B * 100 + S)
        x = torch.randn(B * S, 3 * H * hd, generator=g).half().to(DEV)
        m = _mask("tail", B, S, g).to(DEV) if masked else None
        got = ops.attn(x, B, S, H, hd, hd ** -0.5, causal=True, key_mask=m).float()
        want = _reference(x, B, S, H, hd, True, m)
        assert torch.allclose(got, want, atol=2e-3, rtol=1e-2), (S, (got - want).abs().max().item())


@pytest.mark.parametrize("hd", [136, 256])
@pytest.mark.parametrize("kind", ["none", "tail", "holes"])
def test_causal_wide_heads(hd, kind):
    """head_dim over 128: pair counts on both sides of 8, one to five query blocks of 128, and
    logits far above the first block's."""
    from cobra_amd import ops

    for B, H in ((1, 3), (3, 3), (11, 1)):
        for S in (129, 255, 257, 600):
            g = torch.Generator().manual_seed(B * 10 + S)
            q, k, v = torch.randn(3, B, S, H, hd, generator=g)
            k *= torch.where(torch.arange(S) >= S // 2, 6.0, 1.0)[None, :, None, None]
            x = torch.stack([q, k, v], 2).reshape(B * S, 3 * H * hd).half().to(DEV)
            m = _mask(kind, B, S, g)
            m = None if m is None else m.to(DEV)
            got = ops.attn(x, B, S, H, hd, hd ** -0.5, causal=True, key_mask=m).float()
            want = _reference(x, B, S, H, hd, True, m)
            # probabilities near 1 on values up to 4: 2^-11 of each, and logits of order 20 whose
            # pre-scaled fp16 queries are off by 2^-11 of them
            assert torch.allclose(got, want, atol=1.6e-2, rtol=2e-2), (B, S, (got - want).abs().max().item())


@pytest.mark.parametrize("hd", [8, 32, 40, 64, 72, 128])
@pytest.mark.parametrize("pairs", [37, 1800, 3600])
def test_causal_short(hd, pairs):
    """Up to 128 tokens, few and many (sequence, head) pairs: both kernels of the dispatch, all
    workgroup sizes, with and without a mask; logits raised over the sequence, so that later tiles
    lie above earlier ones."""
    from cobra_amd import ops

    B, H = (pairs // 4, 4) if pairs > 40 else (pairs, 1)
    for S in (1, 32, 33, 64, 65, 96, 97, 127, 128):
        g = torch.Generator(device=DEV).manual_seed(S + pairs)
        x = torch.randn(B, S, 3, H, hd, generator=g, device=DEV)
        x[:, S // 2:, 1] *= 3.0
        x = x.reshape(B * S, 3 * H * hd).half()
        cpu = torch.Generator().manual_seed(S)
        for kind in ("none", "tail", "holes"):
            m = _mask(kind, B, S, cpu)
            m = None if m is None else m.to(DEV)
            got = ops.attn(x, B, S, H, hd, hd ** -0.5, causal=True, key_mask=m).float()
            want = _reference(x, B, S, H, hd, True, m)
            # probabilities near 1 on values up to 4, logits of order 10 (pre-scaled fp16 queries)
            assert torch.allclose(got, want, atol=1e-2, rtol=1e-2), (S, kind, (got - want).abs().max().item())


@pytest.mark.parametrize("hd", [64, 96, 128])
@pytest.mark.parametrize("B,H", [(1, 7), (3, 3), (13, 5), (100, 3)])
def test_causal_many_pairs_of_wide_heads(hd, B, H):
    """The two ways of dealing pairs to the XCDs (heads of whole cache lines, others), one to
    three query blocks."""
    from cobra_amd import ops

    for S in (130, 257, 600):
        g = torch.Generator().manual_seed(B * 100 + S + hd)
        x = torch.randn(B * S, 3 * H * hd, generator=g).half().to(DEV)
        got = ops.attn(x, B, S, H, hd, hd ** -0.5, causal=True).float()
        want = _reference(x, B, S, H, hd, True, None)
        assert torch.allclose(got, want, atol=2e-3, rtol=1e-2), (S, (got - want).abs().max().item())


@pytest.mark.parametrize("hd", [24, 32, 40, 64])
@pytest.mark.parametrize("kind", ["none", "tail", "holes"])
def test_causal_few_long_sequences(hd, kind):
    """At most one workgroup per CU, on both sides of the lengths where the kernel changes, with
    logits that rise over the sequence."""
    from cobra_amd import ops

    B, H = 2, 3
    for S in (511, 512, 513, 777, 2047, 2048, 2500):
        g = torch.Generator(device=DEV).manual_seed(S + hd)
        x = torch.randn(B, S, 3, H, hd, generator=g, device=DEV)
        x[:, S // 2:, 1] *= 3.0
        x = x.reshape(B * S, 3 * H * hd).half()
        m = _mask(kind, B, S, torch.Generator().manual_seed(S))
        m = None if m is None else m.to(DEV)
        got = ops.attn(x, B, S, H, hd, hd ** -0.5, causal=True, key_mask=m).float()
        want = _reference(x, B, S, H, hd, True, m)
        # probabilities near 1 on values up to 4, logits of order 10 (pre-scaled fp16 queries)
        assert torch.allclose(got, want, atol=1e-2, rtol=1e-2), (S, (got - want).abs().max().item())
