"""The 64 x 64 and 128 x 128 tile products (tile_gemm.hip) at the sizes where they can go
wrong: each product in each tile and ring, named, over every count of K slabs around the ring's depth
(test_product_*); and, in what tile the rule picks, extents around a tile, the batch sizes at which
it changes the tile, and the weight gradient."""
import pytest
import torch

import oracle as O
from _gpu import DEV, check, need_gpu, rel_fro, stream
from test_gpu_kernels import bf16_ulps, ns_emul_step
from test_gpu_linear import _gemm_dw, _inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    return need_gpu()


# K of A = X X^T is the wide extent: 1 to 10 slabs of 64; K of the other two products is the
# narrow extent
@pytest.mark.parametrize("rows,cols", [(40, 64 * j - 3) for j in range(1, 11)] + [(64 * j + 1, 40) for j in range(1, 5)] +
                         [(64, 64), (65, 65), (128, 192), (191, 513), (320, 257)])
def test_iterations_vs_emulation_small(L, rows, cols):
    """One and two iterations of a few small matrices against the float64 emulation of the
    rounding scheme (as test_newton_schulz_iterations_vs_emulation, whose bounds these are)."""
    from muon_sr_amd.muon import newton_schulz, NS_COEFFS
    a, b, c = NS_COEFFS
    torch.manual_seed(rows + cols)
    G = (torch.randn(3, rows, cols, device=DEV) * 1e-3).to(torch.bfloat16)
    wide = (lambda t: t.mT) if rows > cols else (lambda t: t)
    prev = G
    for k in range(2):
        X = newton_schulz(G, steps=k + 1)
        emu = ns_emul_step(wide(prev).contiguous(), k == 0, a, b, c)
        u = bf16_ulps(wide(X), emu)
        big = emu.abs() >= 0.25 * emu.pow(2).mean().sqrt()
        assert u[big].max().item() <= 2, (k, u[big].max().item())
        assert rel_fro(wide(X), emu) <= 5e-4, k
        prev = X


@pytest.mark.parametrize("batch,rows,cols", [(64, 1000, 1000), (4, 1000, 1000), (48, 500, 1000), (48, 1000, 500),
                                             (300, 500, 1000), (130, 320, 448), (140, 200, 300), (2, 1920, 2048),
                                             (6, 2048, 1920)])
def test_tiles_give_the_same_bits(L, batch, rows, cols):
    """A matrix alone (64-wide tiles, or 128 for the largest) equals the same matrix in a batch
    that takes 128- or 256-wide tiles, bit for bit: each output element is the same chain of
    MFMAs in every tile."""
    from muon_sr_amd.muon import newton_schulz
    gen = torch.Generator(device=DEV)
    gen.manual_seed(batch + rows)
    G = (torch.randn(batch, rows, cols, device=DEV, generator=gen) * 1e-3).to(torch.bfloat16)
    full = newton_schulz(G)
    for i in (0, batch // 2, batch - 1):
        assert torch.equal(full[i:i + 1].view(torch.int16), newton_schulz(G[i:i + 1].clone()).view(torch.int16)), i


# (256, 256): 64-wide tiles, 2 to 10 slabs; 2048 x 2048: 128-wide, a tile per CU; 2304 x 2048:
# 128-wide, two work-groups per CU (each ring of each tile: test_product_w)
@pytest.mark.parametrize("fout,fin,tokens", [(256, 256, 128 * j) for j in range(1, 6)] +
                         [(2048, 2048, 512), (2048, 2048, 640), (2304, 2048, 512), (2048, 2304, 640)])
@pytest.mark.parametrize("mode", [O.NOISE_TRITON, O.NOISE_PHILOX8])
def test_weight_gradient_tiles(L, fout, fin, tokens, mode):
    """The fused weight gradient in the tile of the rule equals the 256-wide diagnostic GEMM followed by
    msr_sr_accum, bit for bit, with padded rows of x and dy."""
    x, dy, acc = _inputs(tokens, fin, fout, tokens + mode, 8)
    a1, a2 = acc.clone(), acc.clone()
    check(L, L.msr_linear_wgrad_sr_accum(a1.data_ptr(), x.data_ptr(), fin + 8, dy.data_ptr(), fout + 8, tokens, fin, fout,
                                         77, 0, mode, None, stream()), "fused")
    dw = _gemm_dw(L, x, dy, tokens, fin, fout)
    check(L, L.msr_sr_accum(a2.data_ptr(), dw.data_ptr(), 0, fout * fin, 77, 0, mode, None, stream()), "sr_accum")
    assert torch.equal(a1.view(torch.int16), a2.view(torch.int16))


# ---------------------------------------------------------------------------
# each product in each tile and ring; 1 to 9 slabs: the start-up of fewer slabs than stages, every
# tail, and the loop entered once and twice
# ---------------------------------------------------------------------------

CONFIGS = [(64, 4), (64, 2), (128, 4), (128, 2)]
SLABS = range(1, 10)


def _bf(gen, *shape, std=1.0):
    return (torch.randn(*shape, device=DEV, generator=gen) * std).to(torch.bfloat16)


def _product(L, prod, cfg, p, q, d, dims, alpha=1.0, beta=0.0, diag=0.0, rvec=None, resid=None, seed=0, mode=O.NOISE_PHILOX8):
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    check(L, L.msr_tile_gemm(prod, *cfg, ptr(p), ptr(q), ptr(d), *dims, alpha, beta, diag, ptr(rvec), ptr(resid), seed, mode,
                             stream()), (prod, cfg, dims))


def _within(d, ref, mag, k):
    """d = bf16(x) with x a chain of k fp32 multiply-adds (and a few more operations) whose terms' magnitudes sum
    to `mag`: |x - ref| <= e = (k + 8) 2^-24 mag, and half a bf16 ulp of x (at most 2^-8 |x|)."""
    e = (k + 8) * 2.0 ** -24 * mag
    assert bool(((d.double() - ref).abs() <= e + 2.0 ** -8 * (ref.abs() + e) + 1e-38).all())
    return e


def _same(x, y):
    return torch.equal(x.view(torch.int16), y.view(torch.int16))


@pytest.mark.parametrize("cfg", CONFIGS)
@pytest.mark.parametrize("slabs", SLABS)
def test_product_a(L, cfg, slabs):
    """A = X X^T: against float64, exactly symmetric, its residuals, and the 256-wide GEMM's bits (K
    padded with zeros to its multiple of 128)."""
    gen = torch.Generator(device=DEV).manual_seed(slabs)
    m, k = 256, 64 * slabs
    x = _bf(gen, 2, m, k)
    d, resid = torch.empty(2, m, m, device=DEV, dtype=torch.bfloat16), torch.empty(2, m, device=DEV)
    _product(L, 0, cfg, x, None, d, (2, m, m, k), alpha=0.75, resid=resid)
    X = x.double()
    ref, mag = 0.75 * X @ X.mT.contiguous(), 0.75 * X.abs() @ X.abs().mT.contiguous()
    e = _within(d, ref, mag, k)
    assert _same(d, d.mT.contiguous())
    diag = lambda t: t.diagonal(dim1=1, dim2=2)  # noqa: E731
    assert bool(((diag(d).double() + resid.double() - diag(ref)).abs() <= diag(e)).all())
    kp = -(-k // 128) * 128
    xp = torch.zeros(2, m, kp, device=DEV, dtype=torch.bfloat16)
    xp[:, :, :k] = x
    w = torch.empty_like(d)
    check(L, L.msr_gemm_nt(xp.data_ptr(), kp, m * kp, xp.data_ptr(), kp, m * kp, None, m, m * m, w.data_ptr(), m, m * m, m, m,
                           kp, 2, 0.75, 0.0, 0.0, stream()), "gemm")
    assert _same(d, w)


@pytest.mark.parametrize("slabs", SLABS)
def test_product_b(L, slabs):
    """B' = c A A + b A + a I with the diagonal corrected: each configuration that the extent (64 per
    slab) allows against float64 and against the others, bit for bit."""
    gen = torch.Generator(device=DEV).manual_seed(slabs)
    m = 64 * slabs
    s = _bf(gen, 2, m, m, std=m ** -0.5)
    p = (s.float() + s.float().mT).to(torch.bfloat16).contiguous()
    rho = torch.randn(2, m, device=DEV, generator=gen) * 1e-3
    c, b, a = 2.0315, -4.7750, 3.4445
    A, eye = p.double(), torch.eye(m, device=DEV, dtype=torch.float64)
    corr = rho.double() * (b + 2 * c * A.diagonal(dim1=1, dim2=2))
    ref = c * A @ A + b * A + a * eye + torch.diag_embed(corr)
    mag = c * A.abs() @ A.abs() + abs(b) * A.abs() + a * eye + torch.diag_embed(corr.abs() + rho.double().abs() * 10)
    first = None
    for cfg in CONFIGS:
        if m % cfg[0]:
            continue
        d, resid = torch.empty_like(p), torch.empty(2, m, device=DEV)
        _product(L, 1, cfg, p, None, d, (2, m, m, m), alpha=c, beta=b, diag=a, rvec=rho, resid=resid)
        e = _within(d, ref, mag, m)
        assert _same(d, d.mT.contiguous())
        dd, rr = d.diagonal(dim1=1, dim2=2).double(), ref.diagonal(dim1=1, dim2=2)
        assert bool(((dd + resid.double() - rr).abs() <= e.diagonal(dim1=1, dim2=2)).all()), cfg
        first = first or (d, resid)
        assert _same(d, first[0]) and torch.equal(resid, first[1]), cfg


@pytest.mark.parametrize("slabs", SLABS)
@pytest.mark.parametrize("n", [128, 384])
def test_product_x(L, slabs, n):
    """X' = alpha (B' X + bf16(r) X): as test_product_b."""
    gen = torch.Generator(device=DEV).manual_seed(slabs + n)
    m = 64 * slabs
    p, q = _bf(gen, 2, m, m), _bf(gen, 2, m, n)
    r = torch.randn(2, m, device=DEV, generator=gen)
    P, Q, R = p.double(), q.double(), r.to(torch.bfloat16).double()[:, :, None]
    ref, mag = 1.25 * (P @ Q + R * Q), 1.25 * (P.abs() @ Q.abs() + (R * Q).abs())
    first = None
    for cfg in CONFIGS:
        if m % cfg[0]:
            continue
        d = torch.empty_like(q)
        _product(L, 2, cfg, p, q, d, (2, m, n, m), alpha=1.25, rvec=r)
        _within(d, ref, mag, m)
        first = d if first is None else first
        assert _same(d, first), cfg


@pytest.mark.parametrize("cfg", CONFIGS)
@pytest.mark.parametrize("slabs", SLABS)
def test_product_w(L, cfg, slabs):
    """The weight gradient's SR accumulation against the 256-wide GEMM (tokens padded with zeros to its
    multiple of 128) followed by msr_sr_accum, bit for bit."""
    gen = torch.Generator(device=DEV).manual_seed(slabs)
    fout, fin, k = 256, 512, 64 * slabs
    kp = -(-k // 128) * 128
    x, dy = torch.zeros(kp, fin, device=DEV, dtype=torch.bfloat16), torch.zeros(kp, fout, device=DEV, dtype=torch.bfloat16)
    x[:k], dy[:k] = _bf(gen, k, fin), _bf(gen, k, fout, std=1e-2)
    acc = _bf(gen, fout, fin, std=0.1)
    for mode in (O.NOISE_TRITON, O.NOISE_PHILOX8):
        a1, a2 = acc.clone(), acc.clone()
        _product(L, 3, cfg, dy, x, a1, (1, fout, fin, k), seed=77, mode=mode)
        dw = _gemm_dw(L, x, dy, kp, fin, fout)
        check(L, L.msr_sr_accum(a2.data_ptr(), dw.data_ptr(), 0, fout * fin, 77, 0, mode, None, stream()), "sr_accum")
        assert _same(a1, a2)


def test_product_arguments(L):
    x = torch.zeros(256, 256, device=DEV, dtype=torch.bfloat16)
    y, v = torch.zeros_like(x), torch.zeros(256, device=DEV)
    call = lambda prod, tile, stages, m, n, k, d=y, r=v: L.msr_tile_gemm(  # noqa: E731
        prod, tile, stages, x.data_ptr(), x.data_ptr(), d.data_ptr(), 1, m, n, k, 1.0, 0.0, 0.0,
        None if r is None else r.data_ptr(), v.data_ptr(), 0, 1, stream())
    assert call(0, 64, 4, 256, 256, 256) == 0
    assert call(0, 128, 4, 192, 192, 256) == 1001     # not a multiple of the tile
    assert call(0, 64, 4, 256, 256, 100) == 1001
    assert call(0, 64, 3, 256, 256, 256) == 1001
    assert call(0, 32, 4, 256, 256, 256) == 1001
    assert call(0, 64, 4, 256, 128, 256) == 1001      # not square
    assert call(2, 64, 4, 256, 256, 128) == 1001      # the residuals' term needs k = m
    assert call(2, 64, 4, 256, 256, 256, r=None) == 1001
    assert call(4, 64, 4, 256, 256, 256) == 1001
    assert call(0, 64, 4, 256, 256, 256, d=x) == 1005
