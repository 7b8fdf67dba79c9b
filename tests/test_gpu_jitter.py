"""Race check of the decoupled look-back under perturbed timing: with
OSM_FLAG_TIMING_JITTER every workgroup sleeps a pseudo-random 0-13 us (a hash
of its index and the launch) before it publishes its aggregate and before it
combines the words it read, so tiles finish and publish in orders the normal
schedule rarely produces, and checkpoint tiles are often late.  Every entry
point must give the same bits as without the delays, and no look-back wait may
give up (the autouse fixture reads the fault word after each test).  The
reference runs its tiles in one serial loop (sdpc_kernel.py:2006) and has no
such race."""
import pytest
import torch

from helpers import (assert_close_fp32, assert_close_grad, inputs, oracle_backward, oracle_forward, oracle_ttt,
                     to_dev)
from orthossm_amd import cheby_ema_backward, cheby_ema_forward, cheby_ema_ttt
from orthossm_amd import ops

pytestmark = pytest.mark.gpu


def twice(fn):
    """fn() without and with the jitter flag, each result cloned."""
    outs = []
    for on in (False, True):
        old = ops.set_timing_jitter(on)
        try:
            res = fn()
            torch.cuda.synchronize()
            outs.append([t.clone() for t in (res if isinstance(res, (tuple, list)) else (res,))])
        finally:
            ops.set_timing_jitter(old)
    return outs


def assert_same(a, b):
    for i, (x, y) in enumerate(zip(a, b)):
        assert torch.equal(x, y), f"result {i} differs under timing jitter"


@pytest.mark.parametrize("B,S,H,hd,K,dyn", [
    (1, 40_000, 8, 64, 8, False),     # 512-token tiles, past a 64-tile checkpoint group
    (2, 5_000, 8, 64, 8, True),       # dynamic lambda: 256-token tiles, A and B words
    (2, 3_000, 3, 5, 12, False),      # one-lane geometry, Clenshaw form
])
def test_forward_bits_unchanged(dev, B, S, H, hd, K, dyn):
    d = to_dev(inputs(B, S, H, hd, K, seed=S + K, dynamic=dyn), dev)
    init = torch.randn(B, H * hd, device=dev) * 0.3
    a, b = twice(lambda: cheby_ema_forward(d["x"], d["coeffs"], d["damping"], d["lam"], g=d.get("g"),
                                           ema_init=init, return_state=True))
    assert_same(a, b)


def test_jitter_delays_take_effect(dev):
    """The flag reaches the kernels: the delays lengthen a launch (measured on
    MI355X: 81-86 against 46-51 us for this shape)."""
    d = to_dev(inputs(1, 40_000, 8, 64, 8, seed=1), dev)

    def best(on):
        old = ops.set_timing_jitter(on)
        try:
            ts = []
            for _ in range(6):
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                a.record()
                cheby_ema_forward(d["x"], d["coeffs"], d["damping"], d["lam"])
                b.record()
                torch.cuda.synchronize()
                ts.append(a.elapsed_time(b) * 1e3)
            return min(ts[1:])
        finally:
            ops.set_timing_jitter(old)

    plain, jittered = best(False), best(True)
    assert jittered > plain + 10.0, (plain, jittered)


def test_ttt_bits_unchanged(dev):
    d = to_dev(inputs(2, 9_000, 8, 64, 8, seed=71), dev)
    xb = d["x"].to(torch.bfloat16)
    a, b = twice(lambda: cheby_ema_ttt(xb, d["coeffs"], d["damping"], d["lam"]))
    assert_same(a, b)


def test_backward_bits_unchanged(dev):
    d = to_dev(inputs(2, 8_000, 8, 64, 8, seed=72), dev)
    out = cheby_ema_forward(d["x"], d["coeffs"], d["damping"], d["lam"])
    go = torch.randn(out.shape, device=dev, generator=torch.Generator(device=dev).manual_seed(73))
    a, b = twice(lambda: cheby_ema_backward(d["x"], d["coeffs"], d["damping"], d["lam"], out, go, need_init=True))
    assert_same(a, b)


@pytest.mark.parametrize("B,S,H,hd,clamp_tile", [
    (2, 9000, 8, 64, 128),       # the clamp in the first tile
    (1, 9000, 4, 64, 1040),      # four look-back words per thread, the clamp inside a group
    (3, 6000, 7, 48, 2064),      # tiles drawn by ticket
])
def test_table_forward_bits_unchanged(dev, B, S, H, hd, clamp_tile):
    d = to_dev(inputs(B, S, H, hd, 8, seed=S + H), dev)
    init = torch.linspace(-3, 3, B * H * hd, device=dev).view(B, H * hd)
    a, b = twice(lambda: ops.cheby_ema_lut_forward(d["x"], d["coeffs"], n_heads=H, ema_init=init, clamp_tile=clamp_tile,
                                                   ema_momentum=0.999))
    assert_same(a, b)


@pytest.mark.parametrize("B,S,H,hd,dyn", [
    (1, 9000, 1, 64, False),     # one lane-block: its tiles rotate over all eight XCDs
    (3, 5000, 1, 48, True),      # three, of 48 lanes
    (3, 4000, 3, 64, False),     # nine: one more than the XCDs
])
def test_chains_across_xcds(dev, B, S, H, hd, dyn):
    """Lane-block counts off the multiples of 8, whose tiles wait on words
    published on other XCDs: the oracle's values, and the same bits under
    jitter, in the forward, the TTT and the backward."""
    inp = inputs(B, S, H, hd, 8, seed=S, dynamic=dyn)
    d = to_dev(inp, dev)
    go = torch.randn(B, S, H * hd, generator=torch.Generator().manual_seed(S)).to(dev)
    args = (d["x"], d["coeffs"], d["damping"], d["lam"])

    def step():
        out, fin = cheby_ema_forward(*args, g=d.get("g"), return_state=True)
        t_out, t_grad = cheby_ema_ttt(*args, g=d.get("g"))
        gx, gc, _ = cheby_ema_backward(*args, out, go, g=d.get("g"))
        return out, fin, t_out, t_grad, gx, gc

    a, b = twice(step)
    assert_same(a, b)
    want, _ = oracle_forward(inp)
    assert_close_fp32(a[0].cpu(), want)
    assert_close_fp32(a[2].cpu(), want)
    G, _, _ = oracle_ttt(inp)
    assert_close_grad(a[3].cpu(), G, what="ttt gradient")
    wx, wc, _ = oracle_backward(inp, go.cpu().numpy(), out_saved=a[0].cpu().numpy())
    assert_close_grad(a[4].cpu(), wx, what="grad_x")
    assert_close_grad(a[5].cpu(), wc, what="grad_coeffs")


def test_launches_on_several_streams(dev):
    """Launches that wait across XCDs and hold more blocks than the chip has
    places for, on four streams at once: each equals the launch alone, and no
    wait gives up."""
    from orthossm_amd.ops import cheby_ema_lut_forward
    inp = to_dev(inputs(3, 9000, 8, 50, 8, seed=5), dev)
    args = (inp["x"], inp["coeffs"], inp["damping"], inp["lam"])
    go = torch.randn(3, 9000, 400, generator=torch.Generator().manual_seed(6)).to(dev)
    out = cheby_ema_forward(*args)
    calls = (lambda: (cheby_ema_forward(*args),), lambda: cheby_ema_ttt(*args),
             lambda: cheby_ema_backward(*args, out, go)[:2], lambda: cheby_ema_lut_forward(inp["x"], inp["coeffs"], n_heads=8))
    want = [f() for f in calls]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in calls]
    for _ in range(3):
        got = [None] * len(calls)
        for i in range(12):
            with torch.cuda.stream(streams[i % 4]):
                got[i % 4] = calls[(i + i // 4) % 4]()
        torch.cuda.synchronize()
        for i in range(4):
            assert_same(got[i], want[(i + 10) % 4])
    assert ops.workspace_faults() == []
