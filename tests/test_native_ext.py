"""The extension module osm_torch is an accelerator of host time only: without
it, or with one built for another torch or Python, the operators launch through
ctypes, with one warning."""
import ctypes
import warnings

import pytest
import torch

from helpers import inputs, to_dev
from orthossm_amd import _native as nat
from orthossm_amd import cheby_ema_backward, cheby_ema_forward, cheby_ema_ttt, ops


@pytest.fixture
def fresh(monkeypatch):
    """The state before the extension's first use, restored afterwards."""
    monkeypatch.setattr(nat, "_ext", None)
    monkeypatch.setattr(ops, "_ext", None)
    monkeypatch.setattr(ops, "_ext_for", None)
    if ops._raw_stream is None:
        monkeypatch.setattr(ops, "_raw_stream", lambda i: 0)
    return monkeypatch


def _unusable(mp, how):
    if how == "missing":
        mp.setattr(nat, "EXT_PATH", nat.EXT_PATH + ".absent")
    else:
        mp.setattr(torch, "__version__", "0.0.1")


def test_extension_loads_for_this_torch(fresh):
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert nat.load_ext() is not None


@pytest.mark.parametrize("how", ["missing", "other torch"])
def test_without_the_extension_the_ctypes_path_serves(fresh, how):
    _unusable(fresh, how)
    with pytest.warns(RuntimeWarning, match="through ctypes"):
        assert ops._fast() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")      # once
        assert ops._fast() is None
    assert isinstance(nat.load(), ctypes.CDLL)


@pytest.mark.gpu
def test_ctypes_path_gives_the_same_bits(dev, fresh):
    d = to_dev(inputs(2, 700, 4, 32, 8, seed=3), dev)
    args = (d["x"], d["coeffs"], d["damping"], d["lam"])

    def calls():
        out = cheby_ema_forward(*args)
        return out, *cheby_ema_ttt(*args), *cheby_ema_backward(*args, out, torch.ones_like(out), need_init=True)

    want = calls()
    assert ops._ext is not None
    fresh.setattr(nat, "_ext", None)
    fresh.setattr(ops, "_ext_for", None)
    _unusable(fresh, "missing")
    with pytest.warns(RuntimeWarning):
        got = calls()
    for g, w in zip(got, want):
        assert torch.equal(g, w)
