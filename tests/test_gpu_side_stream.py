"""A multi-kernel layer that is refused leaves nothing running: the shared
expert's branch on the library's side stream must not start before everything
that a call can be refused for has been looked at."""
import pytest
import torch

from moe_cases import CONFIGS, Built, reduced

pytestmark = pytest.mark.gpu


def _layer(**spec):
    import zeromoe_amd as Z

    Z.init()
    b = Built(reduced(CONFIGS["c5"], S=16, H=1024, F=512, F_shared=512, router_gemv=False), seed=7)
    L = b.layer()
    for k, v in spec.items():
        setattr(L, k, v)
    return L, torch.from_numpy(b.x).cuda(), torch.from_numpy(b.logits).cuda()


BAD = [dict(n_groups=128), dict(gating=3), dict(gating=-1)]


@pytest.mark.parametrize("spec", BAD, ids=str)
def test_refused_layer_writes_nothing(spec):
    L, x, lg = _layer(**spec)
    ws = L.workspace(16, x.device)
    out = torch.full((16, L.H), 7.0, device="cuda")
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError, match="zm_router"):
        L.forward(x, lg, out=out)
    torch.cuda.synchronize()  # every stream of the device, the library's own among them
    assert not ws.any() and (out == 7.0).all()


@pytest.mark.parametrize("spec", BAD, ids=str)
def test_refused_layer_leaves_a_capture_whole(spec):
    """A refused call inside a capture adds nothing to it: the capture ends
    (an unjoined fork would fail it) and the graph does what is left in it."""
    bad, x, lg = _layer(**spec)
    good, _, _ = _layer()
    bad.workspace(16, x.device)
    eager = good.forward(x, lg)[0].clone()
    out = torch.empty_like(eager)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        with pytest.raises(RuntimeError, match="zm_router"):
            bad.forward(x, lg, out=out)
        good.forward(x, lg, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        assert torch.equal(out, eager)
        good.forward(x, lg)


def test_spec_the_fused_kernel_takes_still_runs():
    """The fused decode kernel ignores a group count it cannot split by."""
    L, x, lg = _layer(n_groups=128)
    ref, _, _ = _layer(n_groups=0)
    assert torch.equal(L.forward(x[:1], lg[:1])[0], ref.forward(x[:1], lg[:1])[0])
