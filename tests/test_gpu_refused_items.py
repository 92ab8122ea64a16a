"""A tensor that the library refuses in the middle of a step: the earlier ones are stepped, it and
the later ones keep their values and the later ones their step, as with one launch per tensor."""
import pytest
import torch

from _gpu import DEV, need_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def L():
    return need_gpu()


def _adamw(ps):
    from muon_sr_amd import TritonAdamW
    return TritonAdamW(ps, lr=0.01)


def _central(ps):
    from muon_sr_amd import TritonAdamW
    return TritonAdamW(ps, lr=0.01, centralization=1.0)


def _eight_bit(ps):
    from muon_sr_amd import TritonAdamW8bit
    return TritonAdamW8bit(ps, lr=0.01, min_8bit_size=6000)


def _muon(ps):
    from muon_sr_amd import TritonMuonSR
    return TritonMuonSR(ps)


@pytest.mark.parametrize("make", [_adamw, _central, _eight_bit, _muon])
@pytest.mark.parametrize("bad", [0, 2, 3])
def test_refused_tensor(make, bad):
    from muon_sr_amd._lib import MuonSRLibraryError
    torch.manual_seed(bad)
    shapes = [(64, 96), (50, 96), (64, 96), (50, 96)]   # 6144 and 4800 elements: both kinds of the 8-bit optimizer
    ps = []
    for i, s in enumerate(shapes):
        n = s[0] * s[1]
        flat = torch.randn(n + 64, device=DEV).bfloat16()
        p = torch.nn.Parameter(flat[:n].view(s))
        # the refused one's gradient overlaps the parameter in part
        p.grad = flat[64:n + 64].view(s) if i == bad else torch.randn_like(p) * 1e-3
        ps.append(p)
    before = [p.detach().clone() for p in ps]
    opt = make(ps)
    with pytest.raises(MuonSRLibraryError, match="overlap"):
        opt.step()
    assert [not torch.equal(p, b) for p, b in zip(ps, before)] == [i < bad for i in range(4)]
    assert [opt.state[p].get("step", 0) for p in ps] == [int(i <= bad) for i in range(4)]
    ps[bad].grad = torch.randn_like(ps[bad]) * 1e-3   # the next step takes them all
    opt.step()
    assert all(not torch.equal(p, b) for p, b in zip(ps, before))
    assert [opt.state[p]["step"] for p in ps] == [2 if i <= bad else 1 for i in range(4)]
