"""GPU checks of the projection GEMM where tiles, k-tiles and 16-byte chunks end.

Every tile size of the dispatch is reached (small grids take 64 x 64 tiles, larger ones up to
256 x 256), with M, N and K on both sides of a tile, K down to one 8-element chunk and not a
multiple of the 64-wide k-tile, residuals and outputs in both widths, bf16, GELU and row
masks.  Reference: float64 torch on the same 16-bit values.  Tolerances: fp32 outputs
`sqrt(K) 2^-22` of the largest output (fp32 sums of exact products, in another order); 16-bit
outputs one unit of roundoff (2^-11, bf16 2^-8) of the value on top.
"""

import pytest
import torch

from _gpu_util import DEV

pytestmark = pytest.mark.gpu


def _check(M, N, K, dtype=torch.float16, out_fp32=False, resid=None, gelu=False, mask=None):
    from cobra_amd import ops

    g = torch.Generator().manual_seed(M * 31 + N * 7 + K)
    a = torch.randn(M, K, generator=g).to(dtype).to(DEV)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype).to(DEV)
    b = torch.randn(N, generator=g).to(DEV)
    r = None if resid is None else torch.randn(M, N, generator=g).to(resid).to(DEV)
    rm = None if mask is None else (torch.rand(M, generator=g) < 0.6).to(DEV)
    got = ops.linear(a, w, b, gelu=gelu, out_fp32=out_fp32, resid=r, rmask=rm, mask_branch=mask == "branch")
    want = a.double() @ w.double().t() + b.double()
    if gelu:
        want = torch.nn.functional.gelu(want)
    if mask == "branch":
        want = want * rm[:, None]
    if r is not None:
        want = want + r.double()
    if mask == "resid":
        want = want * rm[:, None]
    unit = 0.0 if out_fp32 else (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8)
    tol = max(1.0, K ** 0.5) * 2.0 ** -22 * want.abs().max().item() + 2e-6 + unit * want.abs()
    err = (got.double() - want).abs()
    assert got.shape == (M, N) and bool((err <= tol).all()), (M, N, K, dtype, (err - tol).max().item())


@pytest.mark.parametrize("K", [8, 16, 56, 64, 72, 128, 136, 200, 264, 1032])
@pytest.mark.parametrize("N", [8, 24, 64, 72, 200, 720])
def test_small_grids(N, K):
    for M in (1, 31, 64, 65, 129, 300):
        _check(M, N, K, out_fp32=True)
    _check(77, N, K)
    _check(77, N, K, dtype=torch.bfloat16)
    _check(130, N, K, out_fp32=True, resid=torch.float32, gelu=True, mask="branch")
    _check(130, N, K, resid=torch.float16, mask="resid")
    print(f"[gemm-edges] N{N} K{K} ok", flush=True)


@pytest.mark.parametrize("M,N,K", [(2049, 1032, 136), (4100, 1024, 512), (8191, 1024, 72), (8200, 3072, 200),
                                   (12321, 1536, 512), (16385, 3072, 64), (70000, 136, 128)])
def test_large_grids(M, N, K):
    _check(M, N, K)
    _check(M, N, K, out_fp32=True, resid=torch.float32)
    _check(M, N, K, dtype=torch.bfloat16, resid=torch.float32)
    print(f"[gemm-edges] {M}x{N}x{K} ok", flush=True)


@pytest.mark.parametrize("M", [12287, 12288, 12289, 16384, 16385, 32767, 32768, 32769, 32831, 49153, 70001])
def test_many_rows_of_128_to_384(M):
    """Both sides of the line where 128 -> 384 columns take the kernel that keeps W in LDS, and of
    whole rounds of its blocks."""
    _check(M, 384, 128)
    _check(M, 384, 128, dtype=torch.bfloat16)
    _check(M, 384, 128, out_fp32=True)
    _check(M, 384, 128, gelu=True)
    _check(M, 384, 128, mask="branch")
    print(f"[gemm-edges] {M}x384x128 ok", flush=True)


@pytest.mark.parametrize("N", [1, 7, 9, 65, 130])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_columns_not_in_groups_of_8(N, dtype):
    """The register-staged kernel, which takes N % 8 != 0: both residual and output widths, GELU,
    both row masks, K with and without a ragged k-tile, and grids for its 64- and 128-row tiles."""
    for M, K in ((1, 8), (65, 72), (300, 200), (70001 if N <= 65 else 33000, 64)):
        for out_fp32 in (False, True):
            _check(M, N, K, dtype=dtype, out_fp32=out_fp32)
            _check(M, N, K, dtype=dtype, out_fp32=out_fp32, resid=dtype, gelu=True)
            _check(M, N, K, dtype=dtype, out_fp32=out_fp32, resid=torch.float32, mask="branch")
            _check(M, N, K, dtype=dtype, out_fp32=out_fp32, resid=dtype, mask="resid")
    print(f"[gemm-edges] N{N} {dtype} ok", flush=True)


@pytest.mark.parametrize("K", [8, 72, 200])
def test_rows_keep_to_themselves(K):
    """An infinite row of A gives one non-finite output row: the zeros past the end of K are
    zeros on both operands, not the next row's head."""
    from cobra_amd import ops

    a = torch.ones(130, K, device=DEV, dtype=torch.float16)
    a[50] = float("inf")
    w = torch.ones(72, K, device=DEV, dtype=torch.float16)
    out = ops.linear(a, w, None, out_fp32=True)
    finite = torch.isfinite(out).all(1)
    assert not finite[50] and finite.sum().item() == 129
    assert bool((out[finite] == K).all())


def test_gelu_tail():
    """GELU far into the negative tail, where 1 + erf cancels: relative to 64 bits."""
    from cobra_amd import ops

    v = torch.linspace(-5.0, 5.0, 1024, device=DEV).half()
    a = torch.zeros(1024, 8, device=DEV, dtype=torch.float16)
    a[:, 0] = v
    w = torch.zeros(8, 8, device=DEV, dtype=torch.float16)
    w[:, 0] = 1.0
    got = ops.linear(a, w, None, gelu=True, out_fp32=True)[:, 3].double()
    want = v.double() * 0.5 * torch.special.erfc(-v.double() * 0.5 ** 0.5)
    assert bool(((got - want).abs() <= 4e-6 * want.abs() + 1e-12).all())


def test_gelu_far_tail_of_fp32_sums():
    """GELU of sums with 24 bits, to -9: the exponent v^2 / 2 is rounded twice (2^-24 of it each),
    and the rest of the formula is good to 2e-6."""
    from cobra_amd import ops

    v = torch.linspace(-9.0, 9.0, 8192, dtype=torch.float64, device=DEV)
    hi = v.half()
    lo = ((v - hi.double()) * 4096.0).half()
    a = torch.zeros(8192, 8, device=DEV, dtype=torch.float16)
    a[:, 0], a[:, 1] = hi, lo
    w = torch.zeros(8, 8, device=DEV, dtype=torch.float16)
    w[:, 0], w[:, 1] = 1.0, 2.0 ** -12
    v = (hi.double() + lo.double() * 2.0 ** -12).float().double()  # the sum, rounded once
    got = ops.linear(a, w, None, gelu=True, out_fp32=True)[:, 3].double()
    want = v * 0.5 * torch.special.erfc(-v * 0.5 ** 0.5)
    assert bool(((got - want).abs() <= (v * v * 2.0 ** -24 + 2e-6) * want.abs()).all())
