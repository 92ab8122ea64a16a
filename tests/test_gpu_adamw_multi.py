"""Many tensors per launch of the bf16-moment AdamW steps (msr_adamw_multi, both forms)."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from _gpu import check, dev_to_u16, need_gpu, stream, u16_to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    return need_gpu()


def _tensor(rng, n, kind):
    """p, g, m, v as bf16 bits.  kind 0: values of a run (all fast); 1: zeros among them; 2: moments
    at both ends of the fast branch's ranges; 3: as 2 with non-finite gradients (8-bit form only)."""
    p = rng.standard_normal(n) * 0.02
    g = rng.standard_normal(n) * 1e-3
    m = rng.standard_normal(n) * 1e-4
    v = (rng.standard_normal(n) * 1e-3) ** 2
    if kind == 1:
        z = rng.random(n) < 0.7
        g[z], m[z], v[z] = 0.0, 0.0, 0.0
    if kind >= 2:
        at = rng.random(n) < 0.02     # a few per wave of 512 elements: some waves stay fast
        e = rng.integers(-120, 50, n)
        g[at] = np.ldexp(rng.standard_normal(n), e)[at]
        m[at] = np.ldexp(rng.standard_normal(n), rng.integers(-110, 50, n))[at]
        v[at] = np.ldexp(np.abs(rng.standard_normal(n)), rng.integers(-130, 60, n))[at]
    u = [O.f32_to_bf16_rne(x.astype(np.float32)) for x in (p, g, m, v)]
    if kind == 3:
        u[1][rng.integers(0, n, max(1, n // 300))] = 0x7F80
        u[1][rng.integers(0, n, max(1, n // 300))] = 0xFFC0
    return u


def _expect(form, t, hyper, seed, mode):
    lr, b1, b2, eps, wd, bc1, bc2 = hyper
    ns = [O.NoiseSpec(mode, seed, k) for k in range(3)]
    if form == 0:
        return O.adamw_bf16(*t, lr, b1, b2, eps, wd, bc1, bc2, *ns)
    r = O.adamw8bit(*t, None, None, None, None, 256, False, lr, b1, b2, eps, wd, bc1, bc2, *ns)
    return r[0], r[1], r[2]


# a tile is 2048 elements; 56 tensors per launch
SIZES = [1, 7, 8, 9, 511, 512, 513, 2047, 2048, 2049, 4096, 5003, 3, 6000]


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("mode", [O.NOISE_TRITON, O.NOISE_PHILOX8])
@pytest.mark.parametrize("count,kind,eps", [(14, 0, 1e-8), (70, 1, 1e-10), (14, 2, 1e-8), (14, 3, 1e-8), (14, 0, 1e-30)])
def test_multi_vs_oracle(L, form, mode, count, kind, eps):
    """Every tensor of a call against the oracle, bit for bit: sizes around a tile, more tensors
    than one launch takes, aligned and misaligned ones, values on both sides of the fast
    branch's ranges (and eps = 1e-30, which leaves them altogether), a bias correction per tensor."""
    from muon_sr_amd import _lib
    if form == 0 and kind == 3:
        kind = 2   # without the mask, non-finite gradients give NaNs whose payloads are the machine's
    rng = np.random.default_rng(100 * form + 10 * mode + kind)
    lr, b1, b2, wd = 1e-3, 0.9, 0.999, 0.01
    items, want, dev = [], [], []
    for i in range(count):
        n = SIZES[i % len(SIZES)]
        t = _tensor(rng, n, kind)
        step = 1 + i % 5
        bc = (1 - b1 ** step, (1 - b2 ** step) ** 0.5) if form == 0 else (1 - b1 ** step, 1 - b2 ** step)
        seed = (0x9E3779B9 * (i + 1)) & 0xFFFFFFFF
        want.append(_expect(form, t, (lr, b1, b2, eps, wd, *bc), seed, mode))
        off = i % 3 == 2
        d = []
        for x in t:
            y = u16_to_dev(np.concatenate([np.zeros(1, np.uint16), x])) if off else u16_to_dev(x)
            d.append(y[1:] if off else y)
        dev.append(d)
        items.append(_lib.AdamWItem(d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), d[3].data_ptr(), n, *bc, seed, 0))
    arr = (_lib.AdamWItem * count)(*items)
    check(L, L.msr_adamw_multi(ctypes.addressof(arr), count, form, 0.0, lr, b1, b2, eps, wd, mode, stream()), "multi")
    for i, (d, w) in enumerate(zip(dev, want)):
        for k, x in enumerate((d[0], d[2], d[3])):
            assert np.array_equal(dev_to_u16(x), np.asarray(w[k]).ravel()), (i, d[0].numel(), "pmv"[k])


def test_items_that_share_memory_run_in_order(L):
    """The same tensor twice in one call: the second step starts from the first one's result."""
    from muon_sr_amd import _lib
    rng = np.random.default_rng(5)
    t = _tensor(rng, 3000, 0)
    hyper = (1e-3, 0.9, 0.999, 1e-8, 0.01, 0.1, 0.0316)
    p, m, v = _expect(0, t, hyper, 7, O.NOISE_PHILOX8)
    p, m, v = _expect(0, [p, t[1], m, v], hyper, 8, O.NOISE_PHILOX8)
    d = [u16_to_dev(x) for x in t]
    ptrs = [x.data_ptr() for x in d]
    arr = (_lib.AdamWItem * 2)(*[_lib.AdamWItem(*ptrs, 3000, hyper[5], hyper[6], s, 0) for s in (7, 8)])
    check(L, L.msr_adamw_multi(ctypes.addressof(arr), 2, 0, 0.0, *hyper[:5], O.NOISE_PHILOX8, stream()), "multi")
    for x, w in zip((d[0], d[2], d[3]), (p, m, v)):
        assert np.array_equal(dev_to_u16(x), w)


# threads per row 8 ... 256; one group per thread up to 2048 elements, two beyond
COLS = [8, 16, 64, 72, 128, 136, 512, 520, 1024, 1032, 2048, 2056, 3000, 4096]


@pytest.mark.parametrize("mode", [O.NOISE_TRITON, O.NOISE_PHILOX8])
@pytest.mark.parametrize("strength", [1.0, 0.3])
def test_centralized_equals_centralize_then_step(L, mode, strength):
    """The fused form against msr_centralize_bf16 followed by msr_adamw_bf16_step, bit for bit."""
    from muon_sr_amd import _lib
    rng = np.random.default_rng(3)
    hyper = (1e-3, 0.9, 0.999, 1e-8, 0.01, 0.1, 0.0316)
    items, want, dev = [], [], []
    for i, cols in enumerate(COLS):
        for rows in (1, 3, 70):
            n = rows * cols
            t = _tensor(rng, n, 1 if rows == 3 else 0)
            d, e = [u16_to_dev(x) for x in t], [u16_to_dev(x) for x in t]
            nb = ctypes.c_size_t()
            check(L, L.msr_centralize_workspace_bytes(rows, cols, ctypes.byref(nb)))
            ws = torch.empty(max(1, nb.value), dtype=torch.uint8, device=e[0].device)
            c = torch.empty_like(e[1])
            check(L, L.msr_centralize_bf16(e[1].data_ptr(), c.data_ptr(), rows, cols, strength, ws.data_ptr(), ws.numel(),
                                           stream()), "centralize")
            check(L, L.msr_adamw_bf16_step(e[0].data_ptr(), c.data_ptr(), e[2].data_ptr(), e[3].data_ptr(), n, *hyper,
                                           100 + i, mode, None, stream()), "step")
            want.append(e)
            dev.append(d)
            items.append(_lib.AdamWItem(*[x.data_ptr() for x in d], n, hyper[5], hyper[6], 100 + i, cols))
    arr = (_lib.AdamWItem * len(items))(*items)
    check(L, L.msr_adamw_multi(ctypes.addressof(arr), len(items), 2, strength, *hyper[:5], mode, stream()), "multi")
    for it, d, w in zip(items, dev, want):
        for k in (0, 2, 3):
            assert torch.equal(d[k].view(torch.int16), w[k].view(torch.int16)), (it.n // it.cols, it.cols, "pgmv"[k])
    bad = (_lib.AdamWItem * 1)(_lib.AdamWItem(*[x.data_ptr() for x in dev[0]], 8, 0.1, 0.03, 1, 4104))
    assert L.msr_adamw_multi(ctypes.addressof(bad), 1, 2, strength, *hyper[:5], mode, stream()) == 1001


@pytest.mark.parametrize("octave", range(16, 33))
def test_scaled_quotient_is_correctly_rounded(L, octave):
    """sqrt(v') / sqrt(bias correction) as the fast branch forms it, both scaled by 2^32: every
    denominator of [2^16, 2^32], 16 numerators each over 0 and [2^-43, 2^44], against IEEE division."""
    lo = (127 + octave) << 23
    hi = lo + ((1 << 23) - 1 if octave < 32 else 0)
    counts = torch.zeros(1024, dtype=torch.int32, device="cuda:0")
    check(L, L.msr_fastmath_check(5, lo, hi, counts.data_ptr(), 1024, stream()), "fastmath check")
    assert int(counts.sum().item()) == 0
    assert L.msr_fastmath_check(5, 0x47800000 - 1, 0x47800000, counts.data_ptr(), 1024, stream()) == 1001
    assert L.msr_fastmath_check(5, 0x4F800000, 0x4F800001, counts.data_ptr(), 1024, stream()) == 1001
