"""Matrices of their own in shared launches (msr_muon_each) against one msr_muon_fused_step per
matrix, bit for bit, and the class paths that use them."""
import ctypes

import pytest
import torch

import oracle as O
from _gpu import DEV, check, need_gpu, ptr_array, stream

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    return need_gpu()


def _make(shapes, f32, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda s, std: torch.randn(s, device=DEV, generator=gen).mul(std)  # noqa: E731
    return [dict(g=rnd(s, 1e-3) if f32(i) else rnd(s, 1e-3).bfloat16(), b=rnd(s, 1e-3).bfloat16(), p=rnd(s, 0.02).bfloat16(),
                 seeds=(0x9E3779B9 * (i + 1) & 0xFFFFFFFF, 0x85EBCA6B * (i + 1) & 0xFFFFFFFF)) for i, s in enumerate(shapes)]


def _scale(s):
    return max(1.0, s[0] / s[1]) ** 0.5


def _one_by_one(L, mats, mode):
    from muon_sr_amd.muon import NS_COEFFS
    for m in mats:
        r, c = m["p"].shape
        nb = ctypes.c_size_t(0)
        check(L, L.msr_ns_workspace_bytes(1, r, c, ctypes.byref(nb)))
        ws = torch.empty(nb.value, dtype=torch.uint8, device=DEV)
        check(L, L.msr_muon_fused_step(ptr_array([m["g"].data_ptr()]), int(m["g"].dtype == torch.float32),
                                       m["b"].data_ptr(), 0, 1, r, c, 0.95, 1, m["seeds"][0], 5, *NS_COEFFS, None,
                                       ptr_array([m["p"].data_ptr()]), ptr_array([m["seeds"][1]], ctypes.c_uint32), 0.02,
                                       0.01, m.get("scale", _scale((r, c))), mode, None, None, ws.data_ptr(), nb.value, stream()))


def _each(L, mats, mode):
    from muon_sr_amd import _lib
    from muon_sr_amd.muon import NS_COEFFS
    arr = (_lib.MuonMatrix * len(mats))(*[
        _lib.MuonMatrix(m["g"].data_ptr(), m["b"].data_ptr(), m["p"].data_ptr(), *m["p"].shape, *m["seeds"],
                        int(m["g"].dtype == torch.float32), m.get("scale", _scale(m["p"].shape))) for m in mats])
    at, n = ctypes.addressof(arr), len(mats)
    nb = ctypes.c_size_t(0)
    check(L, L.msr_muon_each_workspace_bytes(at, n, ctypes.byref(nb)))
    ws = torch.empty(nb.value, dtype=torch.uint8, device=DEV)
    check(L, L.msr_muon_each(at, n, 0.95, 1, 5, *NS_COEFFS, 0.02, 0.01, mode, ws.data_ptr(), nb.value, stream()))


CASES = {
    "mixed": [(256, 512), (100, 60), (512, 256), (64, 64), (60, 100), (256, 512), (61, 99), (512, 256), (100, 60)],
    "many": [(48, 80)] * 100 + [(80, 48)] * 140,          # more than one prologue and apply launch
    "runs": [(4096, 4096)] * 10 + [(1024, 4096)] * 3,     # more elements than one run takes (8 of 4096 x 4096)
}


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("mode", [O.NOISE_TRITON, O.NOISE_PHILOX8])
def test_each_equals_one_by_one(L, case, mode):
    """Shapes, transposes and gradient types mixed in one list."""
    mk = lambda: _make(CASES[case], lambda i: i % 3 == 1, 7)  # noqa: E731
    x, y = mk(), mk()
    _one_by_one(L, x, mode)
    _each(L, y, mode)
    for i, (u, v) in enumerate(zip(x, y)):
        assert torch.equal(u["b"].view(torch.int16), v["b"].view(torch.int16)), i
        assert torch.equal(u["p"].view(torch.int16), v["p"].view(torch.int16)), i


def test_matrices_that_share_memory_run_in_order(L):
    """The same parameter twice (with momenta of their own): the second step starts from the first."""
    mk = lambda: _make([(128, 192), (128, 192), (192, 128)], lambda i: False, 9)  # noqa: E731
    x, y = mk(), mk()
    x[1]["p"], y[1]["p"] = x[0]["p"], y[0]["p"]
    _one_by_one(L, x, O.NOISE_PHILOX8)
    _each(L, y, O.NOISE_PHILOX8)
    for u, v in zip(x, y):
        assert torch.equal(u["p"].view(torch.int16), v["p"].view(torch.int16))


def test_error_leaves_earlier_parameters_stepped(L):
    """A parameter that is refused stops the step where one launch per parameter would."""
    from muon_sr_amd import TritonMuonSR
    torch.manual_seed(0)
    ps = [torch.nn.Parameter(torch.randn(64, 96, device=DEV).bfloat16()) for _ in range(2)]
    bad = torch.nn.Parameter(torch.randn(96, 64, device=DEV).bfloat16().t())   # not contiguous
    last = torch.nn.Parameter(torch.randn(64, 96, device=DEV).bfloat16())
    for p in (*ps, bad, last):
        p.grad = torch.randn_like(p) * 1e-3
    before = [p.detach().clone() for p in (*ps, bad, last)]
    with pytest.raises(RuntimeError, match="contiguous"):
        TritonMuonSR([*ps, bad, last]).step()
    changed = [not torch.equal(p, b) for p, b in zip((*ps, bad, last), before)]
    assert changed == [True, True, False, False]


def test_scales_of_their_own(L):
    """Matrices of one shape whose scales differ: each is stepped with its own."""
    mk = lambda: _make([(64, 96)] * 5 + [(96, 64)] * 2, lambda i: i == 3, 11)  # noqa: E731
    scales = [1.0, 0.5, 1.0, 0.25, 0.5, 2.0, 1.0]
    x, y = mk(), mk()
    for m, s in zip((*x, *y), scales * 2):
        m["scale"] = s
    _one_by_one(L, x, O.NOISE_PHILOX8)
    _each(L, y, O.NOISE_PHILOX8)
    for i, (u, v) in enumerate(zip(x, y)):
        assert torch.equal(u["p"].view(torch.int16), v["p"].view(torch.int16)), i
