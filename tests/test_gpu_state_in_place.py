"""A recurrent state kept in one buffer: ema_final written to ema_init's memory
(forward, TTT), the gradient of the state likewise (backward), and ema_init a
row of out.  The last tile may end before an earlier tile of the first look-back
group has resolved its carry, so those tiles take the first tile's published
state; timing jitter moves the tiles against each other.  The carry composes
in another order than with buffers apart: equal to rounding."""
import pytest
import torch

from helpers import inputs, to_dev
from orthossm_amd import cheby_ema_backward, cheby_ema_forward, cheby_ema_ttt, ops

pytestmark = pytest.mark.gpu


def close(got, want):
    for g, w in zip(got, want):
        scale = w.double().abs().max().item()
        assert (g.double() - w.double()).abs().max().item() <= 1e-5 * scale


@pytest.fixture(params=[False, True], ids=["", "jitter"])
def jitter(request):
    old = ops.set_timing_jitter(request.param)
    yield
    ops.set_timing_jitter(old)


@pytest.mark.parametrize("B,S,H,hd,dyn", [
    (2, 3000, 8, 64, False),     # 16 lane-blocks: one XCD each
    (1, 9000, 4, 64, False),     # four, few with many tiles: groups of 32
    (3, 4000, 3, 50, True),      # nine, dynamic lambda
    (4, 16384, 8, 64, False),    # 512-token tiles
    (1, 100, 2, 32, False),      # one tile
])
def test_state_in_place(dev, jitter, B, S, H, hd, dyn):
    d = to_dev(inputs(B, S, H, hd, 8, seed=S + H, dynamic=dyn), dev)
    args, kw = (d["x"], d["coeffs"], d["damping"], d["lam"]), dict(g=d.get("g"))
    init = torch.linspace(-0.9, 0.9, B * H * hd, device=dev).view(B, H * hd)
    want = cheby_ema_forward(*args, ema_init=init, return_state=True, **kw)
    s = init.clone()
    got = cheby_ema_forward(*args, ema_init=s, state_out=s, return_state=True, **kw)
    assert got[1] is s
    close(got, want)
    s = init.clone()
    close(cheby_ema_ttt(*args, ema_init=s, state_out=s, return_state=True, **kw),
          cheby_ema_ttt(*args, ema_init=init, return_state=True, **kw))
    go = torch.randn(B, S, H * hd, generator=torch.Generator().manual_seed(S)).to(dev)
    s = init.clone()
    close(cheby_ema_backward(*args, want[0], go, grad_state=s, grad_init_out=s, **kw),
          cheby_ema_backward(*args, want[0], go, grad_state=init, need_init=True, **kw))
    if B == 1:
        out = torch.zeros(1, S, H * hd, device=dev)
        out[0, -1] = init[0]
        close([cheby_ema_forward(*args, ema_init=out[0, -1:], out=out, **kw)], want[:1])
