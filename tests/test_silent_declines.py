"""The forms that stand in for others (joined projections, the fused block step) give way in
silence to what they don't take, but never to a kernel that failed (CPU, fake backends)."""

import sys
import types
import warnings

import pytest
import torch

import mingru_amd
from mingru_amd import DeltaMinGRU, GivensMinGRU, MinGRU, MinGRUBlock, SignedMinGRU, hip_scans
from mingru_amd import min_gru as mg

BACKEND = "mingru_amd.hip_scans"


def _fake(monkeypatch, mode, **impls):
    fake = types.ModuleType(BACKEND)
    fake.ScanFallback, fake.KernelFailure = hip_scans.ScanFallback, hip_scans.KernelFailure
    fake.available = lambda: True
    fake.SCAN_IMPLS = {}
    fake.delta_joined_reason = lambda **kw: None
    fake.angle_joined_reason = lambda *a: None
    fake.block_step_reason = lambda *a: None
    for name, f in impls.items():
        setattr(fake, name, f)
    monkeypatch.setitem(sys.modules, BACKEND, fake)
    monkeypatch.setattr(mingru_amd, "hip_scans", fake, raising=False)
    monkeypatch.setenv("MINGRU_SCAN", "hip")
    if mode == "auto":  # as on a GPU tensor
        monkeypatch.setattr(mg, "_resolve_scan_mode", lambda is_cuda: "auto")
    monkeypatch.setattr(mg, "_warned_joined_failure", False)


def _raise(exc):
    def impl(*a, **kw):
        raise exc
    return impl


LAYERS = [
    (lambda: MinGRU(4, 6), "gate_scan_packed_impl",
     dict(mingru_gate_scan_impl=lambda k, h, h0: k)),
    (lambda: SignedMinGRU(4, 6), "gate_scan_packed_impl",
     dict(signed_gate_scan_impl=lambda s, z, h, h0, **kw: s)),
    (lambda: GivensMinGRU(4, 16), "angle_joined_scan_impl",
     dict(angle_gated_scan_impl=lambda th, u, gm, z, *a, **kw: z)),
    (lambda: DeltaMinGRU(4, 8, n_heads=2, chunk_size=2), "delta_heads_impl",
     dict(delta_scan_impl=lambda Q, K, V, beta, H0, **kw: (V[..., 0, :], H0))),
]


@pytest.mark.parametrize("layer", range(len(LAYERS)))
def test_joined_kernel_failure_follows_the_mode(monkeypatch, layer):
    build, joined, separate = LAYERS[layer]
    m, x = build(), torch.randn(2, 5, 4)
    failed = _raise(hip_scans.KernelFailure("launch failed"))
    _fake(monkeypatch, "hip", **{joined: failed}, **separate)
    with pytest.raises(RuntimeError, match="MINGRU_SCAN=hip.*launch failed"):
        m(x)
    _fake(monkeypatch, "auto", **{joined: failed}, **separate)
    with pytest.warns(UserWarning, match="launch failed"):
        y = m(x)
    with warnings.catch_warnings():  # once
        warnings.simplefilter("error")
        torch.testing.assert_close(m(x), y)
        _fake(monkeypatch, "auto", **{joined: _raise(hip_scans.ScanFallback("not taken"))},
              **separate)
        torch.testing.assert_close(m(x), y)  # outside its envelope: silent
    _fake(monkeypatch, "hip", **{joined: _raise(hip_scans.ScanFallback("not taken"))}, **separate)
    torch.testing.assert_close(m(x), y)


@pytest.mark.parametrize("mode", ["auto", "hip"])
@pytest.mark.parametrize("exc", [RuntimeError("mg_step_gate failed: status 2"),
                                 torch.OutOfMemoryError("out of memory")])
def test_block_step_failure_is_raised(monkeypatch, mode, exc):
    """As the layers' own step kernels: a launch that fails, or memory that runs out."""
    _fake(monkeypatch, mode, block_step_impl=_raise(exc),
          gate_step_impl=lambda kind, p0, *a: p0)
    m, x = MinGRUBlock(8, 2), torch.randn(2, 8)
    with pytest.raises(type(exc), match=str(exc)):
        m.step(x, None)
    _fake(monkeypatch, mode, block_step_impl=_raise(hip_scans.ScanFallback("not taken")),
          gate_step_impl=lambda kind, p0, *a: p0)
    m.step(x, None)


def test_the_funnel_tells_a_failure_from_a_decline():
    with pytest.raises(hip_scans.KernelFailure, match="scan HIP kernel failed: status 2"):
        hip_scans._funnel("scan", _raise(RuntimeError("status 2")))
    with pytest.raises(hip_scans.ScanFallback) as info:
        hip_scans._funnel("scan", _raise(hip_scans.ScanFallback("not taken")))
    assert type(info.value) is hip_scans.ScanFallback


@pytest.mark.parametrize("block", [
    lambda: MinGRUBlock(4, (1 << 18) + 1),  # rows of more than 2^20 elements
    lambda: MinGRUBlock(4, 0, mixer="delta", mixer_kwargs=dict(n_heads=1, d_k=65, d_v=4)),
    lambda: MinGRUBlock(4, 0, mixer="delta", mixer_kwargs=dict(n_heads=1, nh=6)),
])
def test_block_step_declines_what_its_entries_refuse(monkeypatch, block):
    """The C entries' own limits are declined before them, in silence."""
    m = block()
    plan = mg._block_step_plan(m)
    if plan is None:
        return
    kind, ln1, proj, delta, ln2, mlp = plan
    width = 4 if delta is None else delta[0] * delta[2] * delta[3]
    with pytest.raises(hip_scans.ScanFallback, match="limit"):
        hip_scans.block_step_impl(kind, torch.zeros(1, 4), ln1, proj, torch.zeros(1, width), None,
                                  delta, ln2, mlp)
