"""The 64 x 64 and 128 x 128 tile products (tile_gemm.hip) at the sizes where they can go
wrong: every count of K slabs around the ring's depth, extents around a tile, the batch
sizes at which the rule changes the tile, and the weight gradient in each tile."""
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
# 128-wide, two work-groups per CU
@pytest.mark.parametrize("fout,fin,tokens", [(256, 256, 128 * j) for j in range(1, 6)] +
                         [(2048, 2048, 512), (2048, 2048, 640), (2304, 2048, 512), (2048, 2304, 640)])
@pytest.mark.parametrize("mode", [O.NOISE_TRITON, O.NOISE_PHILOX8])
def test_weight_gradient_tiles(L, fout, fin, tokens, mode):
    """The fused weight gradient in each tile equals the 256-wide diagnostic GEMM followed by
    msr_sr_accum, bit for bit, with padded rows of x and dy."""
    x, dy, acc = _inputs(tokens, fin, fout, tokens + mode, 8)
    a1, a2 = acc.clone(), acc.clone()
    check(L, L.msr_linear_wgrad_sr_accum(a1.data_ptr(), x.data_ptr(), fin + 8, dy.data_ptr(), fout + 8, tokens, fin, fout,
                                         77, 0, mode, None, stream()), "fused")
    dw = _gemm_dw(L, x, dy, tokens, fin, fout)
    check(L, L.msr_sr_accum(a2.data_ptr(), dw.data_ptr(), 0, fout * fin, 77, 0, mode, None, stream()), "sr_accum")
    assert torch.equal(a1.view(torch.int16), a2.view(torch.int16))
