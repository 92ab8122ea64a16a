"""Many tensors per launch of the 8-bit step (msr_adamw8bit_multi), in every block size of the
fast kernel and beside tensors that it does not take."""
import ctypes

import numpy as np
import pytest

import oracle as O
from _gpu import check, dev_to_u16, need_gpu, np_to_dev, stream, u16_to_dev
from test_gpu_kernels import qtable_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    return need_gpu()


def _state(rng, n, block, kind):
    """p, g (bf16 bits), codes and block scales.  kind 0: values of a run; 1: zero gradients and
    zero blocks; 2: extreme scales and non-finite gradients in a few places (exact branch)."""
    nb = -(-n // block)
    p = O.f32_to_bf16_rne((rng.standard_normal(n) * 0.02).astype(np.float32))
    g = (rng.standard_normal(n) * 1e-3).astype(np.float32)
    s1, s2 = rng.integers(0, 256, n).astype(np.uint8), rng.integers(0, 256, n).astype(np.uint8)
    a1 = (np.abs(rng.standard_normal(nb)) * 1e-3).astype(np.float32)
    a2 = (rng.standard_normal(nb).astype(np.float32) * 1e-3) ** 2
    if kind == 1:
        z = rng.random(n) < 0.8
        g[z] = 0.0
        a1[rng.random(nb) < 0.5] = 0.0
    g = O.f32_to_bf16_rne(g)
    if kind == 2:
        g[rng.integers(0, n, max(1, n // 1500))] = 0x7F80
        g[rng.integers(0, n, max(1, n // 1500))] = 0xFFC1
        a1[rng.integers(0, nb, max(1, nb // 20))] = np.float32(2.0) ** rng.integers(-100, 30)
        a2[rng.integers(0, nb, max(1, nb // 20))] = np.float32(2.0) ** rng.integers(-120, 70)
    return p, g, s1, s2, a1, a2


SIZES = [1, 63, 511, 512, 513, 1024, 4096 + 77, 9000, 65, 1536]   # a chunk is 512 elements


@pytest.mark.parametrize("block", [32, 64, 128, 256, 512, 2048])
@pytest.mark.parametrize("mode,kind,count", [(O.NOISE_PHILOX8, 0, 60), (O.NOISE_TRITON, 1, 10), (O.NOISE_PHILOX8, 2, 10)])
def test_multi_vs_oracle(L, block, mode, kind, count):
    """Every tensor of a call against the oracle, bit for bit; every fourth one is misaligned (the
    general kernel)."""
    from muon_sr_amd import _lib
    rng = np.random.default_rng(block + 10 * kind)
    q1, q2 = O.create_dynamic_map(True), O.create_dynamic_map(False)
    d1, d2, qt = np_to_dev(q1), np_to_dev(q2), qtable_dev(L)
    hyper = (3e-4, 0.9, 0.95, 1e-10, 0.01, 1 - 0.9 ** 3, 1 - 0.95 ** 3)
    items, want, dev = [], [], []
    for i in range(count):
        n = SIZES[i % len(SIZES)]
        t = _state(rng, n, block, kind)
        seed = (0x9E3779B9 * (i + 3)) & 0xFFFFFFFF
        want.append(O.adamw8bit(*t, q1, q2, block, True, *hyper, O.NoiseSpec(mode, seed)))
        off = i % 4 == 3
        cat = (lambda x: np.concatenate([np.zeros(1, x.dtype), x])) if off else (lambda x: x)
        d = [u16_to_dev(cat(t[0])), u16_to_dev(cat(t[1])), np_to_dev(cat(t[2])), np_to_dev(cat(t[3])), np_to_dev(t[4]),
             np_to_dev(t[5])]
        if off:
            d[:4] = [x[1:] for x in d[:4]]
        dev.append(d)
        items.append(_lib.Adam8Item(*[x.data_ptr() for x in d], n, seed, 0))
    arr = (_lib.Adam8Item * count)(*items)
    lr, b1, b2, eps, wd, bc1, bc2 = hyper
    check(L, L.msr_adamw8bit_multi(ctypes.addressof(arr), count, d1.data_ptr(), d2.data_ptr(), qt.data_ptr(), block, lr,
                                   b1, b2, eps, wd, bc1, bc2, mode, stream()), "multi")
    for i, (d, w) in enumerate(zip(dev, want)):
        at = (i, d[0].numel(), block)
        assert np.array_equal(dev_to_u16(d[0]), w[0]), at
        assert np.array_equal(d[2].cpu().numpy(), w[1]) and np.array_equal(d[3].cpu().numpy(), w[2]), at
        for x, y in ((d[4], w[3]), (d[5], w[4])):
            assert np.array_equal(x.cpu().numpy().view(np.uint32), y.view(np.uint32)), at
