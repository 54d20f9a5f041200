"""What the fused decode step of a block refuses on the host, before any launch (CPU)."""

import pytest
import torch
from torch import nn

from mingru_amd import MinGRUBlock, hip_scans
from mingru_amd import min_gru as mg

D, B = 16, 3

# An edit of a block and the mixer it applies to.  Each leaves a module whose layers don't
# fit together, which torch refuses when it runs them one by one.
EDITS = {
    "norm1": ("log", lambda b: setattr(b, "norm1", nn.LayerNorm((1, D)))),
    "norm2": ("log", lambda b: setattr(b, "norm2", nn.LayerNorm(8))),
    "norm bias": ("log", lambda b: setattr(b.norm2, "bias", nn.Parameter(torch.zeros(8)))),
    "mlp wider": ("log", lambda b: b.mlp.__setitem__(0, nn.Linear(D, 128))),
    "mlp narrower": ("signed", lambda b: b.mlp.__setitem__(0, nn.Linear(D, 32))),
    "mlp in": ("signed", lambda b: b.mlp.__setitem__(0, nn.Linear(32, 64))),
    "mlp out": ("log", lambda b: b.mlp.__setitem__(3, nn.Linear(64, 32))),
    "gate rows": ("log", lambda b: setattr(b.mingru, "linear_h", nn.Linear(D, 12))),
    "gate columns": ("signed", lambda b: setattr(b.mingru, "linear_s", nn.Linear(20, D))),
    "bias": ("signed", lambda b: setattr(b.mingru.linear_z, "bias", nn.Parameter(torch.zeros(8)))),
    "weight rank": ("log", lambda b: setattr(b.mingru.linear_z, "weight",
                                             nn.Parameter(torch.zeros(D * D)))),
    "out_proj": ("delta", lambda b: setattr(b.mingru, "out_proj", nn.Linear(32, D))),
    "out_proj rows": ("delta", lambda b: setattr(b.mingru, "out_proj", nn.Linear(D, 20))),
    # The joined rows add up to the same sum with k and v exchanged.
    "heads": ("delta", lambda b: (b.mingru.linear_k.__setitem__(0, nn.Linear(D, 8)),
                                  b.mingru.linear_v.__setitem__(0, nn.Linear(D, 24)))),
    "beta": ("delta", lambda b: b.mingru.linear_beta.__setitem__(0, nn.Linear(D, 1))),
}


def _step(block):
    kind, *rest = mg._block_step_plan(block)
    ln1, proj, delta, ln2, mlp = rest
    h = torch.zeros(B, D if kind != "delta" else delta[0] * delta[2] * delta[3])
    return hip_scans.block_step_impl(kind, torch.zeros(B, D), ln1, proj, h, None, delta, ln2, mlp)


@pytest.mark.parametrize("edit", EDITS)
def test_disagreeing_widths_are_refused(edit):
    mixer, change = EDITS[edit]
    block = MinGRUBlock(D, 4, mixer=mixer, mixer_kwargs={"n_heads": 2} if mixer == "delta" else None)
    with pytest.raises(hip_scans.ScanFallback, match="GPU tensors"):
        _step(block)
    change(block)
    with pytest.raises(hip_scans.ScanFallback, match="shape"):
        _step(block)


@pytest.mark.parametrize("mixer", ["log", "delta"])
def test_state_and_decay_of_another_shape_are_refused(mixer):
    block = MinGRUBlock(D, 0, mixer=mixer, mixer_kwargs={"n_heads": 2} if mixer == "delta" else None)
    kind, ln1, proj, delta, ln2, mlp = mg._block_step_plan(block)
    width = D if delta is None else delta[0] * delta[2] * delta[3]
    x = torch.zeros(B, D)
    for h, gamma in ((torch.zeros(B, width - 1), None), (torch.zeros(B + 1, width), None),
                     (torch.zeros(B, width), torch.zeros(B, 1))):
        with pytest.raises(hip_scans.ScanFallback, match="shape"):
            hip_scans.block_step_impl(kind, x, ln1, proj, h, gamma, delta, ln2, mlp)


@pytest.mark.parametrize("d,b,taken", [
    (4096, 1, True), (4096, 2, False), (8192, 1, False), (3072, 4, True), (3072, 5, False),
    (2048, 8, True), (2048, 9, False), (1024, 48, True), (1024, 49, False), (256, 192, True),
    (256, 193, False), (18, 2, False)])
def test_sizes_that_the_layers_run_faster_are_declined(d, b, taken):
    """Padded sequences times the square of the width bound the kernels' work, beside the
    bounds on the input; the message tells the size's refusal from the CPU tensors'."""
    meta = lambda *s: torch.empty(*s, device="meta")  # noqa: E731
    ln, pair = (meta(d), meta(d), 1e-5), (meta(d, d), meta(d))
    with pytest.raises(hip_scans.ScanFallback, match="GPU tensors" if taken else "width"):
        hip_scans.block_step_impl("mingru", meta(b, d), ln, [pair] * 2, meta(b, d), None, None, None,
                                  None)


def test_a_size_that_is_declined_plans_nothing(monkeypatch):
    """The dispatch looks at the input's size, type and layout before it walks the block's
    modules, and takes the layers; for another input it goes on to the plan."""
    plans = []
    real = mg._block_step_plan
    monkeypatch.setenv("MINGRU_SCAN", "hip")
    monkeypatch.setattr(hip_scans, "available", lambda: True)
    monkeypatch.setattr(mg, "_block_step_plan", lambda b: plans.append(1) or real(b))
    block = MinGRUBlock(D, 0)
    for n, planned in ((257, []), (3, [1])):
        assert mg._dispatch_block_step(block, torch.zeros(n, D), None, None) is None
        assert plans == planned
    assert mg._dispatch_block_step(block, torch.zeros(3, 2, D)[:, 1], None, None) is None
    assert mg._dispatch_block_step(block.half(), torch.zeros(3, D).half(), None, None) is None
    assert plans == [1]
