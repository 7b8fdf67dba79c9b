"""The entry points under HIP graph capture (torch.cuda.CUDAGraph): a captured
forward, TTT step, backward and full path replay several times, with eager launches of
the same entry points and host synchronisations in between, and every replay
equals the eager result bit for bit.  The workspaces of the capture stream
are created by a warm-up on that stream before capture, so the graphs hold
only the library's kernels (no memset nodes); launches keep their state in
the workspace (epoch, look-back words), not on the host."""
import pytest
import torch

from helpers import inputs, to_dev
from orthossm_amd import cheby_ema_backward, cheby_ema_forward, cheby_ema_ttt, ops

pytestmark = pytest.mark.gpu


def _capture(fn, stream):
    """Warm fn up on `stream`, then capture it there; returns the graph."""
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(2):
            fn()
    stream.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        fn()
    torch.cuda.synchronize()
    return g


@pytest.mark.parametrize("dynamic", [False, True])
def test_forward_graph_replays_match_eager(dev, dynamic):
    d = to_dev(inputs(2, 5000, 8, 64, seed=31, dynamic=dynamic), dev)
    other = to_dev(inputs(1, 3000, 8, 64, seed=32, dynamic=dynamic), dev)
    init = torch.randn(2, 512, device=dev) * 0.3
    want, want_fin = cheby_ema_forward(d["x"], d["coeffs"], d["damping"], d["lam"], g=d.get("g"), ema_init=init,
                                       return_state=True)
    out = torch.empty_like(want)
    fin = torch.empty_like(want_fin)

    def step():
        cheby_ema_forward(d["x"], d["coeffs"], d["damping"], d["lam"], g=d.get("g"), ema_init=init, out=out,
                          return_state=True, state_out=fin)

    g = _capture(step, torch.cuda.Stream())
    for i in range(4):
        out.fill_(float("nan"))
        g.replay()
        # eager work of the same entry point on the default stream in between
        cheby_ema_forward(other["x"], other["coeffs"], other["damping"], other["lam"], g=other.get("g"))
        torch.cuda.synchronize()
        assert torch.equal(out, want), f"replay {i}"
        assert torch.equal(fin, want_fin), f"replay {i} ema_final"


def test_ttt_graph_replays_match_eager(dev):
    inp = inputs(2, 3000, 8, 64, seed=33)
    d = to_dev(inp, dev)
    xb = d["x"].to(torch.bfloat16)
    want_out, want_grad = cheby_ema_ttt(xb, d["coeffs"], d["damping"], d["lam"])
    out = torch.empty_like(want_out)
    grad = torch.empty_like(want_grad)

    def step():
        cheby_ema_ttt(xb, d["coeffs"], d["damping"], d["lam"], out=out, grad_out=grad)

    g = _capture(step, torch.cuda.Stream())
    for i in range(4):
        grad.zero_()
        g.replay()
        cheby_ema_ttt(xb[:1, :1000], d["coeffs"][:1], d["damping"], d["lam"])
        torch.cuda.synchronize()
        assert torch.equal(out, want_out), f"replay {i}"
        assert torch.equal(grad, want_grad), f"replay {i} grad"


def test_backward_graph_replays_match_eager(dev):
    d = to_dev(inputs(2, 4000, 8, 64, seed=34), dev)
    out = cheby_ema_forward(d["x"], d["coeffs"], d["damping"], d["lam"])
    go = torch.randn(out.shape, device=dev, generator=torch.Generator(device=dev).manual_seed(35))
    want = cheby_ema_backward(d["x"], d["coeffs"], d["damping"], d["lam"], out, go, need_init=True)
    gx, gc, gi = (torch.empty_like(t) for t in want)

    def step():
        cheby_ema_backward(d["x"], d["coeffs"], d["damping"], d["lam"], out, go, grad_x_out=gx,
                           grad_coeffs_out=gc, grad_init_out=gi)

    g = _capture(step, torch.cuda.Stream())
    for i in range(4):
        gx.zero_()
        g.replay()
        cheby_ema_backward(d["x"][:1], d["coeffs"][:1], d["damping"], d["lam"], out[:1], go[:1])
        torch.cuda.synchronize()
        for got, w, what in zip((gx, gc, gi), want, ("grad_x", "grad_coeffs", "grad_init")):
            assert torch.equal(got, w), f"replay {i} {what}"


def _three_calls(dev, seed):
    """{name: call} of the forward, TTT and backward on one set of inputs, and
    the same calls on a shape whose workspaces are many times larger."""
    small, big = (to_dev(inputs(B, S, 8, 64, seed=seed), dev) for B, S in ((1, 2000), (8, 16384)))

    def calls(d):
        args = (d["x"], d["coeffs"], d["damping"], d["lam"])
        out = cheby_ema_forward(*args)
        go = torch.ones_like(out)
        return dict(forward=lambda: (cheby_ema_forward(*args),), ttt=lambda: cheby_ema_ttt(*args),
                    backward=lambda: cheby_ema_backward(*args, out, go, need_init=True))

    return calls(small), calls(big)


@pytest.mark.parametrize("name", ["forward", "ttt", "backward"])
@pytest.mark.parametrize("warm", [True, False])
def test_graph_outlives_the_workspace_of_its_stream(dev, name, warm):
    """After a capture, eager calls on the capture stream grow that stream's
    workspace and other tensors take what memory is free; the replays still
    match and touch none of it.  Also for a capture with no call before it."""
    small, big = _three_calls(dev, 41)
    want = [t.clone() for t in small[name]()]
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        if warm:
            small[name]()
            stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            got = small[name]()
        for i in range(3):
            eager = big[name]() if i else small[name]()
            filled = [torch.full((n,), 3.0, device=dev) for n in (1 << 18, 1 << 20, 1 << 22)]
            for t in got:
                t.fill_(float("nan"))
            graph.replay()
            stream.synchronize()
            assert all((f == 3.0).all() for f in filled)
            for g, w in zip(got, want):
                assert torch.equal(g, w), f"replay {i}"
            if i == 0:
                for g, w in zip(eager, want):
                    assert torch.equal(g, w)
    kept = [ws.numel() for key, ws in ops._ws_kept if key[1] == stream.cuda_stream]
    assert sum(kept) <= sum(ws.numel() for key, ws in ops._ws_cache.items() if key[1] == stream.cuda_stream)
    assert ops.workspace_faults() == []


def test_first_use_in_a_capture_leaves_later_eager_calls_right(dev):
    """The engine's fast path with a carried state and the drop-in, first used
    in a capture (seven heads, a momentum of its own): eager calls before any
    replay, on the capture stream and on another, and the replays match."""
    from orthossm_amd import ChebyContextPath, ChebyState, apply_cheby_rkv_v10
    H, hd, S = 7, 12, 50
    torch.manual_seed(1)
    path = ChebyContextPath(H * hd, n_cheby_heads=H, max_degree=4, carry_ema=True).to(dev).eval()
    x = torch.randn(2, S, H * hd, device=dev)
    c = torch.randn(2, H, 4, hd, device=dev) * 0.3
    state = ChebyState(c, torch.zeros_like(c), torch.full((2, H * hd), 0.2, device=dev))

    def step():
        with torch.no_grad():
            path.total_tokens_seen.zero_()
            r = path(x, state)
            return r.out, apply_cheby_rkv_v10(x, c, None, n_heads=H, ema_momentum=0.8125)[0]

    lam = path.ema_base.new_full((H,), 0.8125)
    damp = torch.tensor([0.98 - 0.06 * h / H for h in range(H)], device=dev)
    want = cheby_ema_forward(x, c, damp, lam, nan_policy="zero_u")
    torch.cuda.synchronize()
    cap, other = torch.cuda.Stream(), torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=cap):
        got = step()
    eager = []
    for s in (cap, other):
        with torch.cuda.stream(s):
            eager.append(step())
    torch.cuda.synchronize()
    for out, fast in eager:
        torch.testing.assert_close(fast, want, rtol=1e-5, atol=1e-6)
        assert torch.equal(out, eager[0][0])
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        for g, w in zip(got, eager[0]):
            assert torch.equal(g, w)


def test_full_path_graph_replays_match_eager(dev):
    from orthossm_amd.ops import v10_chunked_ttt
    gen = torch.Generator().manual_seed(36)
    x = torch.randn(2, 900, 256, generator=gen).to(dev)
    c = (torch.randn(2, 4, 8, 64, generator=gen) * 0.3).to(dev)
    m = (torch.randn(2, 4, 8, 64, generator=gen) * 0.01).to(dev)
    mu = torch.tensor(0.85, device=dev)
    want = v10_chunked_ttt(x, c, m, n_heads=4, ema_momentum=mu)
    res = [None]

    def step():
        res[0] = v10_chunked_ttt(x, c, m, n_heads=4, ema_momentum=mu)

    g = _capture(step, torch.cuda.Stream())
    for i in range(4):
        g.replay()
        v10_chunked_ttt(x[:1, :300], c[:1], m[:1], n_heads=4)
        torch.cuda.synchronize()
        for got, w, what in zip(res[0], want, ("out", "coeffs", "momentum")):
            assert torch.equal(got, w), f"replay {i} {what}"


def test_forward_graph_with_other_layouts_on_the_capture_stream(dev):
    # Between replays an eager call of another shape runs on the capture
    # stream, so on the same workspace with another layout (the library
    # clears its look-back words).  The captured launch then reuses the
    # workspace with no host step; the inputs change before every replay, so
    # a look-back word left by an earlier replay (another payload) that
    # matched a later launch's tag would give a wrong result.
    big = [to_dev(inputs(2, 6000, 8, 64, seed=40 + i), dev) for i in range(4)]
    small = to_dev(inputs(1, 700, 8, 64, seed=39), dev)
    xbuf = big[0]["x"].clone()
    c, damp, lam = big[0]["coeffs"], big[0]["damping"], big[0]["lam"]
    out = torch.empty_like(xbuf)
    cap = torch.cuda.Stream()

    def step():
        cheby_ema_forward(xbuf, c, damp, lam, out=out)

    g = _capture(step, cap)
    for i in range(4):
        xbuf.copy_(big[i]["x"])
        want = cheby_ema_forward(xbuf, c, damp, lam)        # default stream, its own workspace
        torch.cuda.synchronize()
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), f"replay {i}"
        with torch.cuda.stream(cap):
            cheby_ema_forward(small["x"][:, : 300 + 100 * i], small["coeffs"], small["damping"], small["lam"])
        torch.cuda.synchronize()
