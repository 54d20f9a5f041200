"""GPU parity of the fused decode step of a residual block (csrc/decode_block.hip).

A no-op hook on the block's norm makes ``MinGRUBlock.step`` run layer by layer, so each
case holds the fused step against the block in float64 and against that step: in fp32 both
are within 2e-6 of float64 (sums of up to 800 terms at 2^-24 each), in bf16 the fused step,
which rounds less often, may be no further off than the layers, plus one rounding (2^-8).
"""

import copy

import pytest
import torch

from mingru_amd import MinGRUBlock, MinGRUStack, hip_scans

pytestmark = pytest.mark.gpu

CASES = [
    # d, B, mixer, its options, MLP expansion; batch tiles 1, 4, 8, 16 and their edges
    (64, 1, "log", {}, 4),
    (200, 3, "log", {"bias": False}, 2),
    (256, 8, "signed", {"coupled": True}, 4),
    (260, 5, "signed", {"decay": "learnable"}, 0),
    (132, 16, "log", {"decay": "fixed"}, 1),
    (64, 4, "delta", {"n_heads": 2, "nh": 2}, 4),
    (200, 9, "delta", {"n_heads": 5, "d_k": 12, "d_v": 20, "decay": "learnable"}, 1),
    (256, 2, "delta", {"n_heads": 4, "bias": False}, 4),
    # Several groups of 16 sequences, the last one partial.
    (128, 17, "signed", {"decay": "learnable"}, 2),
    (64, 70, "delta", {"n_heads": 1}, 1),
]


def _state(case, cuda, dtype, g):
    d, B, mixer, kw, _ = case
    if mixer == "delta":
        h = kw["n_heads"]
        dk = kw.get("d_k", d // h)
        return (0.3 * torch.randn(B, h * dk * kw.get("d_v", dk), generator=g)).to(cuda, dtype)
    x = torch.randn(B, d, generator=g)
    return (x.abs() if mixer == "log" else x).to(cuda, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("given_state", [True, False])
@pytest.mark.parametrize("case", CASES)
def test_block_step(cuda, case, given_state, dtype, monkeypatch):
    d, B, mixer, kw, exp = case
    print(f"[gpu] block step {case} {dtype} state={given_state}", flush=True)
    monkeypatch.setenv("MINGRU_SCAN", "hip")
    torch.manual_seed(3)
    g = torch.Generator().manual_seed(4)
    fused = MinGRUBlock(d, exp, mixer=mixer, mixer_kwargs=kw).to(cuda, dtype).eval()
    layers = copy.deepcopy(fused)
    layers.norm1.register_forward_hook(lambda *a: None)
    x = torch.randn(B, d, generator=g).to(cuda, dtype)
    h = _state(case, cuda, dtype, g) if given_state else None
    dt = torch.rand(B, generator=g).to(cuda, dtype) if kw.get("decay") else None
    calls = []
    real = hip_scans._call
    monkeypatch.setattr(hip_scans, "_call",
                        lambda name, *a: (real(name, *a), calls.append(name)))
    y, s = fused.step(x, h, dt)
    launches = ["mg_step_gate"] if mixer != "delta" else [
        "mg_step_project", "mg_delta_step_heads", "mg_step_project"]
    launches += ["mg_step_project"] * (2 if exp else 0)
    assert calls == launches, "the fused step did not run"
    calls.clear()
    yl, sl = layers.step(x, h, dt)
    assert calls == ["mg_delta_step" if mixer == "delta" else "mg_gate_step"]
    monkeypatch.setenv("MINGRU_SCAN", "eager")
    ref = copy.deepcopy(fused).double()
    yr, sr = ref.step(x.double(), None if h is None else h.double(),
                      None if dt is None else dt.double())
    torch.cuda.synchronize()
    for name, a, b, r in (("x", y, yl, yr), ("state", s, sl, sr)):
        assert a.dtype == b.dtype == dtype and a.shape == b.shape
        off, own = ((t.double() - r).norm() / r.norm().clamp_min(1e-30) for t in (a, b))
        bound = 2e-6 if dtype == torch.float32 else own + 2.0**-8
        assert off <= bound, f"{name}: {off.item():.2e} off float64, layers {own.item():.2e}"


def test_block_step_declines(cuda, monkeypatch):
    """What the fused step does not stand in for runs layer by layer: an active dropout,
    another mixer; and, declined by the backend, a large batch and a sliced input."""
    monkeypatch.setenv("MINGRU_SCAN", "hip")

    def refuse(*a):
        raise AssertionError("the fused step must not run")

    torch.manual_seed(0)
    m = MinGRUBlock(64, 2).to(cuda)
    with monkeypatch.context() as c:
        c.setattr(hip_scans, "block_step_impl", refuse)
        drop = MinGRUBlock(64, 2, dropout=0.1).to(cuda)
        drop.train().step(torch.randn(2, 64, device=cuda), None)
        MinGRUBlock(64, 2, mixer="givens").to(cuda).step(torch.randn(2, 64, device=cuda), None)
    monkeypatch.setattr(hip_scans, "_call", lambda name, *a, r=hip_scans._call: (
        refuse() if name == "mg_step_gate" else r(name, *a)))
    m.step(torch.randn(257, 64, device=cuda), None)
    wide = torch.randn(2, 128, device=cuda)
    y, _ = m.step(wide[:, ::2], None)  # not dense
    monkeypatch.undo()
    torch.testing.assert_close(y, m.step(wide[:, ::2].contiguous(), None)[0], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("mode", ["auto", "hip"])
def test_block_step_of_layers_that_do_not_fit(cuda, mode, monkeypatch):
    """An edited block whose layers disagree raises torch's error, as its forward does."""
    monkeypatch.setenv("MINGRU_SCAN", mode)
    m = MinGRUBlock(64, 2).to(cuda).eval()
    m.mlp[0] = torch.nn.Linear(64, 256).to(cuda)  # wider than mlp[3] reads
    x = torch.randn(2, 64, device=cuda)
    with pytest.raises(RuntimeError, match="shapes cannot be multiplied"):
        m.step(x, None)
    m.mlp[3] = torch.nn.Linear(256, 64).to(cuda)
    y, _ = m.step(x, None)
    torch.testing.assert_close(y, m(x[:, None])[0][:, 0], rtol=1e-5, atol=1e-5)


def test_stack_stream_equals_forward(cuda, monkeypatch):
    """A streamed hybrid stack equals its forward over the sequence."""
    monkeypatch.setenv("MINGRU_SCAN", "hip")
    torch.manual_seed(1)
    m = MinGRUStack(32, 64, 3, mixer=["log", "signed", "delta"],
                    mixer_kwargs={"delta": {"n_heads": 2}}).to(cuda).eval()
    x = torch.randn(3, 150, 32, device=cuda)
    with torch.no_grad():
        y, _ = m(x)
    state = m.init_state()
    for t in range(x.shape[1]):
        out, state = m.step(x[:, t].contiguous(), state)
        assert (out - y[:, t]).abs().max().item() <= 1e-4
