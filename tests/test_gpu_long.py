"""Invariants over a million tokens, as the reference checks its long
streams (finite and |out| <= 1 up to 1M tokens, benchmark_long_context.py:
300-349; NaN/Inf scans over streamed tokens, benchmark_ortho.py:153-205),
plus call-splitting invariants that hold bit for bit:

* the full path (online TTT with Lion over 4096 chunks of 256 tokens) run
  as one call equals the same sequence run as four calls with the
  coefficients and momentum carried from one call to the next (the chunks
  never see the call boundaries); the coefficients stay within the Lion
  bound |c_k| <= max(|c_k(0)|, lr ss_k / (1 - d)), d = lambda - lr wd;
* the forward over 2^20 tokens run as one call equals four calls with the
  EMA state carried, to the fp32 tolerance of the look-back composition.
"""
import numpy as np
import pytest
import torch

from oracle import v10_full as V
from orthossm_amd import cheby_ema_forward
from orthossm_amd.ops import v10_chunked_ttt
from orthossm_amd.synthetic import make_inputs

pytestmark = pytest.mark.gpu


def test_full_path_backward_at_the_last_tokens_of_int32(dev):
    """dL/dx of one lane over 2^31 - 200 tokens in chunks of 2^20: the last
    chunk's end is past what a sum of its start and the chunk length holds.
    x = z = 0, one linear coefficient, dL/dout = 1: dL/dx is (1-mu) gamma times
    the sum of mu^i over the tokens left in the chunk."""
    from orthossm_amd.ops import _v10_backward
    S, chunk, mu = (1 << 31) - 200, 1 << 20, 0.9
    n = (S + chunk - 1) // chunk
    x = torch.zeros(1, S, 1, dtype=torch.bfloat16, device=dev)
    out = torch.zeros(1, S, 1, device=dev)
    hist = torch.zeros(n, 1, 1, 2, 1, device=dev)
    hist[:, :, :, 1] = 1.0
    gx, _ = _v10_backward(x, out, x, hist, torch.ones(1, device=dev).expand(1, S, 1), 1, mu, chunk, False)
    left = torch.arange(3, 0, -1, dtype=torch.float64)
    want = 0.98 * (1.0 - mu ** left)
    for end in (S, S // chunk * chunk, chunk):
        got = gx[0, end - 3:end, 0].double().cpu()
        assert (got - want).abs().max() <= 2.0 ** -8 * want.max(), (end, got, want)

S_LONG = 1 << 20


def test_full_path_million_tokens_split_calls_and_lion_bound(dev):
    H, hd, K = 8, 64, 8
    gen = torch.Generator().manual_seed(123)
    x = torch.randn(1, S_LONG, H * hd, generator=gen).to(dev)
    c0 = (torch.randn(1, H, K, hd, generator=gen) / torch.arange(1, K + 1).view(1, 1, K, 1)).to(dev)
    m0 = torch.zeros_like(c0)
    out, c1, m1 = v10_chunked_ttt(x, c0, m0, n_heads=H, chunk_size=256)
    # the same sequence as four calls of 2^18 tokens, (c, m) carried
    parts = []
    c, m = c0, m0
    q = S_LONG // 4
    for i in range(4):
        o, c, m = v10_chunked_ttt(x[:, i * q:(i + 1) * q], c, m, n_heads=H, chunk_size=256)
        parts.append(o)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all() and out.abs().max().item() <= 1.0
    assert torch.isfinite(c1).all() and torch.isfinite(m1).all()
    assert torch.equal(torch.cat(parts, dim=1), out)
    assert torch.equal(c, c1) and torch.equal(m, m1)
    # Lion: c <- d c + lr ss_k sign(.), so |c| stays within max(|c0|, lr ss_k / (1 - d)).
    lam, ss, lr_scale = V.lion_constants(H, K)
    lr = 0.005 * lr_scale
    d = lam - lr * 0.01
    bound = lr[:, None] * ss[None, :] / (1.0 - d[:, None])            # [H, K]
    got = c1.abs().cpu().numpy()[0]                                   # [H, K, hd]
    start = c0.abs().cpu().numpy()[0]
    # fp32 rounding of each update, damped by d per chunk, and of d and
    # lr ss_k themselves, move the limit by ~1e-4 relative at 1 - d = 5e-4
    lim = np.maximum(start, bound[:, :, None]) * (1 + 1e-3) + 1e-6
    assert (got <= lim).all(), f"max excess {(got - lim).max():.3e}"


@pytest.mark.parametrize("dynamic", [False, True])
def test_forward_million_tokens_split_calls(dev, dynamic):
    inp = make_inputs(1, S_LONG, 512, 8, 8, seed=7, dynamic=dynamic)
    d = {k: v.to(dev) for k, v in inp.items() if v is not None}
    g = d.get("g")
    out, fin = cheby_ema_forward(d["x"], d["coeffs"], d["damping"], d["lam"], g=g, return_state=True)
    q = S_LONG // 4
    state = None
    parts = []
    for i in range(4):
        sl = slice(i * q, (i + 1) * q)
        o, state = cheby_ema_forward(d["x"][:, sl], d["coeffs"], d["damping"], d["lam"],
                                     g=None if g is None else g[:, sl], ema_init=state, return_state=True)
        parts.append(o)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all() and out.abs().max().item() <= 1.0
    split = torch.cat(parts, dim=1)
    # the carry enters through a different composition order: fp32 tolerance
    tol = 1e-5 * out.abs() + 1e-6
    assert ((split - out).abs() <= tol).all()
    assert ((state - fin).abs() <= 1e-5 * fin.abs() + 1e-6).all()
