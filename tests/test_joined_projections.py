"""The joined projections: which layers they stand in for (CPU, a fake backend), and that
the joined form equals the separate one (GPU).

A no-op forward hook on one projection makes a module run its projections separately, so
the GPU cases compare the two forms of one module; the native calls of each are recorded,
so that a joined form that gave way to the separate one does not pass for it.  In fp32 both
compute the same sums in another order and agree to 2e-5 (sums of up to a few thousand terms
at 2^-24 each).  In bf16 the separate form rounds after every eager operation and the joined
one at its kernels' outputs only, so each is held against the module in float64: the joined
form may be 1.5 times as far off as the separate one plus one rounding of the output (2^-8).
It is nearer on average, 0.73 to 1.0 times; the 1.5 is the chance part of outputs with a
handful of entries.
"""

import copy
import ctypes
import importlib
import sys
import types

import pytest
import torch
from torch import nn
from torch.utils._python_dispatch import TorchDispatchMode

import mingru_amd
from mingru_amd import DeltaMinGRU, GivensMinGRU, MinGRU, SignedMinGRU
from mingru_amd import min_gru as mg

BACKEND = "mingru_amd.hip_scans"
HIP_SCANS = importlib.import_module(BACKEND)


def _fake(monkeypatch, calls):
    class FakeFallback(Exception):
        pass

    def joined(kind, P, h0, dt=None, lam=None, *, h0_const=0.0):
        calls.append(("joined", kind, tuple(P.shape), h0 is None))
        return P[..., : P.shape[-1] // (2 if kind == "mingru" else 3)]

    fake = types.ModuleType(BACKEND)
    fake.ScanFallback = FakeFallback
    fake.available = lambda: True
    fake.SCAN_IMPLS = {}
    fake.gate_scan_packed_impl = joined
    fake.mingru_gate_scan_impl = lambda k, h, h0, *a: calls.append(("separate",)) or k
    fake.signed_gate_scan_impl = lambda s, z, h, h0, **kw: calls.append(("separate",)) or s
    monkeypatch.setitem(sys.modules, BACKEND, fake)
    monkeypatch.setattr(mingru_amd, "hip_scans", fake, raising=False)
    monkeypatch.setenv("MINGRU_SCAN", "hip")


class _MyLinear(nn.Linear):
    pass


def test_plain_projections_are_joined(monkeypatch):
    calls = []
    _fake(monkeypatch, calls)
    x = torch.randn(2, 5, 4)
    m = MinGRU(4, 6)
    out = m(x)  # the fake returns the first projection's slice
    assert calls == [("joined", "mingru", (2, 5, 12), True)]
    torch.testing.assert_close(out, m.linear_z(x))
    calls.clear()
    s = SignedMinGRU(4, 6, coupled=True, learnable_h0=True)
    torch.testing.assert_close(s(x), s.linear_s(x))
    assert calls == [("joined", "signed_coupled", (2, 5, 18), False)]


@pytest.mark.parametrize("why", ["hook", "pre_hook", "subclass", "frozen", "half", "no_grad_rows",
                                 "patched_forward", "mixed_bias"])
def test_other_projections_stay_separate(monkeypatch, why):
    calls = []
    _fake(monkeypatch, calls)
    m = MinGRU(4, 6)
    x = torch.randn(2, 5, 4)
    seen = []
    if why == "hook":
        m.linear_h.register_forward_hook(lambda *a: seen.append(1))
    elif why == "pre_hook":
        m.linear_h.register_forward_pre_hook(lambda *a: seen.append(1))
    elif why == "subclass":
        m.linear_h = _MyLinear(4, 6)
    elif why == "frozen":
        m.linear_h.weight.requires_grad_(False)
    elif why == "half":
        m, x = m.double(), x.double()
    elif why == "patched_forward":
        m.linear_h.forward = lambda v: seen.append(1) or nn.functional.linear(
            v, m.linear_h.weight, m.linear_h.bias)
    elif why == "mixed_bias":
        m.linear_h = nn.Linear(4, 6, bias=False)
    if why == "no_grad_rows":
        with torch.no_grad():
            m(x)
    else:
        m(x)
    assert calls == [("separate",)]
    if why in ("hook", "pre_hook", "patched_forward"):
        assert seen == [1]


def _fake_delta(monkeypatch, calls):
    """The fake backend with the delta entry points; the scan keeps the true envelope."""
    _fake(monkeypatch, calls)
    fake = sys.modules[BACKEND]

    def heads(P, H, nh, dk, dv):
        calls.append("heads")
        B, T, _ = P.shape
        return tuple(P.new_zeros(B, H, T, *s) for s in ((dk,), (nh, dk), (nh, dv), (nh,)))

    def scan(Q, K, V, beta, *rest, chunk_size):
        if K.shape[3] * chunk_size > 128:
            raise fake.ScanFallback("nh * chunk_size")
        calls.append("scan")
        return V[..., 0, :], rest[-1]

    fake.delta_heads_impl = heads
    fake.delta_scan_impl = fake.delta_gated_scan_impl = scan
    fake.delta_joined_reason = lambda **kw: HIP_SCANS.delta_joined_reason(
        **dict(kw, is_cuda=True))
    fake.angle_joined_scan_impl = lambda *a: calls.append("joined")
    fake.angle_joined_reason = HIP_SCANS.angle_joined_reason
    return fake


@pytest.mark.parametrize("decay", [None, "learnable"])
def test_delta_heads_stay_separate_under_autocast(monkeypatch, decay):
    """Under autocast the keys are normalised in fp32 and the scan runs in fp32; one joined
    bf16 product would round them and move the whole layer to the bf16 kernels."""
    calls = []
    _fake_delta(monkeypatch, calls)
    m = DeltaMinGRU(8, 8, n_heads=2, decay=decay)
    x, dt = torch.randn(2, 6, 8), torch.rand(2, 6) if decay else None
    m(x, delta_t=dt)
    assert calls == ["heads", "scan"]
    calls.clear()
    kind = torch.get_autocast_dtype("cuda")
    torch.set_autocast_enabled("cuda", True)
    torch.set_autocast_dtype("cuda", torch.bfloat16)
    try:
        m(x, delta_t=dt)
    finally:
        torch.set_autocast_dtype("cuda", kind)
        torch.set_autocast_enabled("cuda", False)
    assert calls == ["scan"]


WIDTHS = {
    # Layers edited to widths that add up to the right sum, or to a multiple of it.
    "mingru": (lambda: MinGRU(4, 6), {"linear_z": (4, 8), "linear_h": (4, 4)}),
    "mingru wider": (lambda: MinGRU(4, 6), {"linear_h": (4, 10)}),
    "signed": (lambda: SignedMinGRU(4, 6), {"linear_s": (4, 5), "linear_h": (4, 7)}),
    "givens": (lambda: GivensMinGRU(4, 16), {"linear_z": (4, 12), "linear_h": (4, 20)}),
    "delta": (lambda: DeltaMinGRU(8, 8, n_heads=2), {"linear_q": (8, 6), "linear_k.0": (8, 10)}),
    "delta beta": (lambda: DeltaMinGRU(8, 8, n_heads=2), {"linear_v.0": (8, 9),
                                                          "linear_beta.0": (8, 1)}),
    "delta lists": (lambda: DeltaMinGRU(8, 8, n_heads=2), {"linear_k.1": (8, 8),
                                                           "linear_v.1": (8, 8)}),
}


@pytest.mark.parametrize("case", WIDTHS)
def test_projections_of_other_widths_stay_separate(monkeypatch, case):
    """Side by side, rows of another split would pass for the right ones; one by one, torch
    refuses them."""
    calls = []
    _fake_delta(monkeypatch, calls)
    build, widths = WIDTHS[case]
    m = build()
    for name, (i, o) in widths.items():
        parent, _, leaf = name.rpartition(".")
        m.get_submodule(parent).add_module(leaf, nn.Linear(i, o))
    monkeypatch.setattr(mg, "_join_linears", lambda *a: calls.append("product") or _real(*a))
    try:
        m(torch.randn(2, 5, m.input_size))
    except (RuntimeError, IndexError):
        pass
    assert "product" not in calls, calls


_real = mg._join_linears


OUTSIDE = {
    # module, delta_t's shape, h_0: what the kernels decline whatever the projection holds.
    "delta microsteps": (lambda: DeltaMinGRU(8, 8, n_heads=2, nh=3), None, None),
    "delta chunk": (lambda: DeltaMinGRU(8, 8, n_heads=2, chunk_size=65, decay="fixed"), (2, 5), None),
    "delta state": (lambda: DeltaMinGRU(8, 8, n_heads=2), None, torch.zeros(2, 1, 32).double()),
    "h0 for every row": (lambda: SignedMinGRU(4, 6), None, torch.zeros(1, 1, 6)),
    "h0 type": (lambda: MinGRU(4, 6), None, torch.ones(2, 1, 6).double()),
    "one gap for every row": (lambda: SignedMinGRU(4, 6, decay="fixed"), (1, 5), None),
    "rounds": (lambda: GivensMinGRU(4, 16, rounds=65), None, None),
    "givens state": (lambda: GivensMinGRU(4, 16), None, torch.zeros(2, 1, 16).double()),
}


@pytest.mark.parametrize("case", OUTSIDE)
def test_a_call_the_kernels_decline_projects_nothing_first(monkeypatch, case):
    """The envelope is asked before the joined product, which would be dropped."""
    calls = []
    _fake_delta(monkeypatch, calls)
    build, gaps, h0 = OUTSIDE[case]
    monkeypatch.setattr(mg, "_join_linears", lambda *a: calls.append("product") or _real(*a))
    m = build()
    try:
        m(torch.randn(2, 5, m.input_size), h0, None if gaps is None else torch.rand(*gaps))
    except RuntimeError as exc:
        assert "MINGRU_SCAN=hip" in str(exc)  # the separate form's seam
    assert "product" not in calls, calls


@pytest.mark.parametrize("d,lanes", [(16, 16), (17, 32), (64, 64)])
def test_delta_heads_stay_inside_one_launch(d, lanes):
    """A launch takes fewer than 2^32 threads: past that many lanes the heads are declined
    before the product, and the C entries refuse them (host checks: nothing is launched)."""
    from mingru_amd import _native

    kw = dict(is_cuda=True, dtype=torch.bfloat16, h0_dtype=torch.float32, d_k=d, d_v=8, nh=1,
              chunk_size=64, n_heads=8)
    tokens = (2**32 - 256) // (8 * lanes)  # of 8 heads
    assert HIP_SCANS.delta_joined_reason(**kw, tokens=tokens) is None
    assert "tokens" in HIP_SCANS.delta_joined_reason(**kw, tokens=tokens + 1)
    lib, one = _native.load(), ctypes.c_void_p(16)
    dims = (1, tokens + 1, 8, 1, d, 8, 1)
    assert lib.mg_delta_heads_fwd(*[one] * 6, *dims, None) == 1
    assert lib.mg_delta_heads_bwd(*[one] * 8, *dims, None) == 1


def test_a_bias_that_broadcasts_stays_separate(monkeypatch):
    calls = []
    _fake(monkeypatch, calls)
    m = MinGRU(4, 6)
    m.linear_z.bias = nn.Parameter(torch.zeros(1))
    m.linear_h.bias = nn.Parameter(torch.zeros(11))
    with pytest.raises(RuntimeError, match="size"):
        m(torch.randn(2, 5, 4))
    assert calls == []


def _pair(cuda, m, dtype):
    joined = m.to(cuda, dtype)
    separate = copy.deepcopy(joined)
    for lin in separate.modules():
        if isinstance(lin, nn.Linear):
            lin.register_forward_hook(lambda *a: None)
    return joined, separate


def _record_native(monkeypatch, calls):
    """Appends (entry, arguments) of every native call that returned."""
    real = HIP_SCANS._call

    def call(name, *args):
        real(name, *args)
        calls.append((name, args))

    monkeypatch.setattr(HIP_SCANS, "_call", call)


def _joined_entries(m, dtype):
    """The native entries of ``m``'s joined form, one call each in a training pass."""
    if isinstance(m, GivensMinGRU):
        return {"mg_angle_scan_joined_fwd", "mg_angle_scan_joined_bwd"}
    if isinstance(m, DeltaMinGRU):
        return {"mg_delta_heads_fwd", "mg_delta_heads_bwd"}
    kind = "bf16" if dtype == torch.bfloat16 else "rows"
    return {f"mg_gate_scan_{kind}_fwd", f"mg_gate_scan_{kind}_bwd"}


def _ran_joined(m, dtype, calls):
    entries = _joined_entries(m, dtype)
    ran = [(name, args) for name, args in calls if name in entries]
    if isinstance(m, (MinGRU, SignedMinGRU)):  # the separate bf16 form's rows lie D apart
        n = 2 if isinstance(m, MinGRU) else 3
        ran = [(name, args) for name, args in ran if args[4] == n * m.hidden_size]
    return sorted(name for name, _ in ran) == sorted(entries)


def _off(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30)).item()


MODULES = [
    # constructor, B, T, time decay
    (lambda: MinGRU(24, 48), 3, 200, False),
    (lambda: MinGRU(40, 33, bias=False, learnable_h0=True), 2, 1100, False),
    (lambda: MinGRU(16, 130, decay="learnable"), 2, 70, True),
    (lambda: SignedMinGRU(24, 48), 1, 1, False),
    (lambda: SignedMinGRU(64, 256, coupled=True, learnable_h0=True), 3, 777, False),
    (lambda: SignedMinGRU(32, 520, decay="fixed"), 2, 2100, True),
    # Head dims of 16-, 32- and 64-lane groups with idle lanes, micro-steps, gated.
    (lambda: DeltaMinGRU(24, 48, n_heads=4, chunk_size=16), 2, 133, False),
    (lambda: DeltaMinGRU(40, 96, n_heads=3, nh=2, d_v=20, bias=False), 3, 200, False),
    (lambda: DeltaMinGRU(64, 192, n_heads=3, nh=2, decay="learnable"), 1, 321, True),
    (lambda: DeltaMinGRU(32, 100, n_heads=2, d_k=50, d_v=9, decay="fixed"), 2, 140, True),
]


# 8x8 Givens blocks join in fp32 only (their kernels are fp32): a wave of 64 planes and
# partial ones, the compiled three rounds and the per-token loop, one- and two-level walks.
GIVENS = [
    (lambda: GivensMinGRU(24, 16), 2, 1, False),
    (lambda: GivensMinGRU(32, 512, decay="learnable"), 2, 70, True),
    (lambda: GivensMinGRU(40, 536, bias=False), 1, 300, False),
    (lambda: GivensMinGRU(24, 64, rounds=2, decay="fixed"), 3, 45, True),
    (lambda: GivensMinGRU(24, 48, rounds=5), 2, 290, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", range(len(MODULES + GIVENS)))
def test_joined_equals_separate(cuda, case, dtype, monkeypatch):
    givens = case >= len(MODULES)
    build, B, T, decay = (MODULES + GIVENS)[case]
    print(f"[gpu] joined projections case={case} {dtype}", flush=True)
    monkeypatch.setenv("MINGRU_SCAN", "hip")
    torch.manual_seed(100 + case)
    joined, separate = _pair(cuda, build(), dtype)
    d = joined.input_size
    x = torch.randn(B, T, d, device=cuda, dtype=dtype)
    dt = torch.rand(B, T, device=cuda, dtype=dtype) if decay else None
    res, ran, calls = [], [], []
    _record_native(monkeypatch, calls)
    for m in (joined, separate):
        calls.clear()
        xi = x.clone().requires_grad_()
        y = m(xi, delta_t=dt) if decay else m(xi)
        gy = torch.randn(y.shape, generator=torch.Generator().manual_seed(9)).to(cuda, dtype)
        grads = torch.autograd.grad(y, [xi, *m.parameters()], gy)
        res.append([y.detach(), *grads])
        ran.append(_ran_joined(m, dtype, calls))
    torch.cuda.synchronize()
    assert ran == [not givens or dtype == torch.float32, False]
    if dtype == torch.float32:
        for i, (a, b) in enumerate(zip(*res)):
            assert a.dtype == b.dtype and a.shape == b.shape
            assert _off(a, b) <= 2e-5, f"output {i}: relative difference {_off(a, b):.2e}"
        return
    monkeypatch.setenv("MINGRU_SCAN", "eager")
    ref = copy.deepcopy(joined).double()
    xi = x.double().requires_grad_()
    y = ref(xi, delta_t=dt.double()) if decay else ref(xi)
    exact = [y.detach(), *torch.autograd.grad(y, [xi, *ref.parameters()], gy.double())]
    for i, (a, b, r) in enumerate(zip(*res, exact)):
        assert a.dtype == b.dtype and a.shape == b.shape
        assert _off(a, r) <= 1.5 * _off(b, r) + 2.0**-8, (
            f"output {i}: joined {_off(a, r):.2e}, separate {_off(b, r):.2e} off float64")


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(MODULES + GIVENS)))
def test_joined_equals_separate_under_autocast(cuda, case, monkeypatch):
    """fp32 modules under bf16 autocast: the joined gates round where the separate ones do
    (their products' outputs; bound as for bf16 modules), and the delta and Givens layers,
    whose separate forms compute their heads in fp32, don't join at all: their outputs are
    the same to the last bit."""
    gates = case < 6
    build, B, T, decay = (MODULES + GIVENS)[case]
    print(f"[gpu] joined projections under autocast case={case}", flush=True)
    monkeypatch.setenv("MINGRU_SCAN", "hip")
    torch.manual_seed(100 + case)
    joined, separate = _pair(cuda, build(), torch.float32)
    x = torch.randn(B, T, joined.input_size, device=cuda)
    dt = torch.rand(B, T, device=cuda) if decay else None
    res, ran, calls = [], [], []
    _record_native(monkeypatch, calls)
    for m in (joined, separate):
        calls.clear()
        xi = x.clone().requires_grad_()
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = m(xi, delta_t=dt) if decay else m(xi)
        gy = torch.randn(y.shape, generator=torch.Generator().manual_seed(9)).to(cuda, y.dtype)
        res.append([y.detach(), *torch.autograd.grad(y, [xi, *m.parameters()], gy)])
        ran.append(_ran_joined(m, torch.bfloat16, calls))
    assert ran == [gates, False]
    monkeypatch.setenv("MINGRU_SCAN", "eager")
    ref = copy.deepcopy(joined).double()
    xi = x.double().requires_grad_()
    y = ref(xi, delta_t=dt.double()) if decay else ref(xi)
    exact = [y.detach(), *torch.autograd.grad(y, [xi, *ref.parameters()], gy.double())]
    for i, (a, b, r) in enumerate(zip(*res, exact)):
        assert a.dtype == b.dtype and a.shape == b.shape
        if gates:
            assert _off(a, r) <= 1.5 * _off(b, r) + 2.0**-8, (
                f"output {i}: joined {_off(a, r):.2e}, separate {_off(b, r):.2e} off float64")
        else:
            assert torch.equal(a, b), f"output {i}"


# fp32 layers whose joined backward could sum in another order than the separate one:
# inputs of one long product against several short ones, weights of a few columns.
PRECISION = [
    (lambda: DeltaMinGRU(256, 256, n_heads=4), 8, 1000),
    (lambda: DeltaMinGRU(256, 256, n_heads=4, nh=2), 4, 1500),
    (lambda: SignedMinGRU(320, 320), 8, 500),
    (lambda: MinGRU(256, 512), 4, 700),
    (lambda: GivensMinGRU(256, 512), 4, 500),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(PRECISION)))
def test_joined_gradients_lose_no_precision(cuda, case, monkeypatch):
    """No fp32 gradient is further from float64 joined than separate.  3% is the chance part:
    the smallest outputs compared have some thousand entries.  (The biases, a handful of
    entries in places, are held by the comparison above.)"""
    build, B, T = PRECISION[case]
    print(f"[gpu] joined precision case={case}", flush=True)
    torch.manual_seed(7 + case)
    joined, separate = _pair(cuda, build(), torch.float32)
    x = torch.randn(B, T, joined.input_size, device=cuda)
    gy = None
    res = []
    for m, mode in ((joined, "hip"), (separate, "hip"), (copy.deepcopy(separate).double(), "eager")):
        monkeypatch.setenv("MINGRU_SCAN", mode)
        xi = x.to(next(m.parameters()).dtype).requires_grad_()
        y = m(xi)
        gy = torch.randn(y.shape, generator=torch.Generator().manual_seed(9)).to(cuda) \
            if gy is None else gy
        names = [n for n, _ in m.named_parameters() if n.endswith("weight")]
        grads = torch.autograd.grad(y, [xi, *(m.get_parameter(n) for n in names)], gy.to(y.dtype))
        res.append(grads)
    for n, a, b, r in zip(["x", *names], *res):
        assert _off(a, r) <= 1.03 * _off(b, r), (
            f"{n}: joined {_off(a, r):.3e}, separate {_off(b, r):.3e} off float64")


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("x_grad,w_grad,b_grad", [(True, True, True), (False, True, False),
                                                  (True, False, False), (False, False, True)])
def test_joined_linears_differentiate(bias, x_grad, w_grad, b_grad):
    """The joined projection's own backward: every layer's gradients, layers of a few
    columns and wide ones in any order, each only where it is asked for."""
    torch.manual_seed(2)
    linears = [nn.Linear(12, n, bias=bias) for n in (70, 64, 3, 80, 1)]
    for m in linears:
        m.weight.requires_grad_(w_grad)
        if bias:
            m.bias.requires_grad_(b_grad)
    x = torch.randn(2, 9, 12, requires_grad=x_grad)
    leaves = [t for t in (x, *(p for m in linears for p in m.parameters())) if t.requires_grad]
    if not leaves:
        return
    P, want = mg._join_linears(x, linears), torch.cat([m(x) for m in linears], -1)
    torch.testing.assert_close(P, want)
    g = torch.randn_like(P)
    for a, b in zip(torch.autograd.grad(P, leaves, g), torch.autograd.grad(want, leaves, g)):
        assert a.shape == b.shape and a.dtype == b.dtype
        torch.testing.assert_close(a, b)


class _Products(TorchDispatchMode):
    """Counts the multiply-adds of matrix products and the reductions run inside."""

    def __init__(self):
        super().__init__()
        self.work = self.sums = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if func.overloadpacket in (torch.ops.aten.mm, torch.ops.aten.addmm_):
            a, b = args[-2:]
            self.work += a.shape[0] * a.shape[1] * b.shape[1]
        self.sums += func is torch.ops.aten.sum.dim_IntList
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("leaf", [True, False])
@pytest.mark.parametrize("how", ["grad", "backward"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_joined_linears_form_what_is_asked_for(how, leaf, dtype, monkeypatch):
    """The input's gradient and, past a size (here: any), each weight's are formed only if
    they are asked for, the biases' if any of them is."""
    monkeypatch.setitem(mg._JOIN_ASK_WORK, dtype, 0)
    torch.manual_seed(4)
    linears = [nn.Linear(12, n, dtype=dtype) for n in (70, 64, 3, 80)]
    x = torch.randn(18, 12, dtype=dtype, requires_grad=True)
    if not leaf:
        x = 2 * x
        x.retain_grad()
    one = 18 * 12 * (70 + 64 + 3 + 80)
    asked = [((linears[1].weight,), 18 * 12 * 64, 0), ((x,), one, 0), ((linears[2].bias,), 0, 1),
             ((linears[0].weight, linears[2].weight), 18 * 12 * (70 + 3), 0),
             ((x, *(m.weight for m in linears)), 2 * one, 0),
             ((x, linears[0].bias, linears[3].weight), one + 18 * 12 * 80, 1)]
    for leaves, work, sums in asked:
        P, want = mg._join_linears(x, linears), torch.cat([m(x) for m in linears], -1)
        g = torch.randn_like(P)
        with _Products() as count:
            if how == "grad":
                got = torch.autograd.grad(P, leaves, g, retain_graph=True)
            else:
                for t in leaves:
                    t.grad = None
                P.backward(g, inputs=list(leaves), retain_graph=True)
                got = [t.grad for t in leaves]
        assert (count.work, count.sums) == (work, sums)
        for a, b in zip(got, torch.autograd.grad(want, leaves, g, retain_graph=True)):
            # bf16: a rounding (2^-8) for each of the separate input gradient's four parts, of
            # magnitude 2, and for their sums.
            torch.testing.assert_close(a, b, **({} if dtype == torch.float32 else
                                                dict(rtol=2.0**-6, atol=2.0**-6)))


def test_small_joined_linears_form_all_weights_or_none():
    """Below that size the weights' gradients are one joined product if any is asked for."""
    linears = [nn.Linear(12, n) for n in (70, 64)]
    x = torch.randn(18, 12, requires_grad=True)
    for leaves, work in (((linears[1].weight,), 18 * 12 * 134), ((linears[0].bias,), 0)):
        P = mg._join_linears(x, linears)
        with _Products() as count:
            torch.autograd.grad(P, leaves, torch.ones_like(P))
        assert count.work == work


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_joined_linears_compile(dtype, monkeypatch):
    """Traced, where the engine can't be asked, the products are torch's own."""
    monkeypatch.setitem(mg._JOIN_ASK_WORK, dtype, 0)
    torch.manual_seed(5)
    linears = [nn.Linear(6, n, dtype=dtype) for n in (66, 2)]
    x = torch.randn(2, 4, 6, dtype=dtype, requires_grad=True)
    leaves = [x, *(p for m in linears for p in m.parameters())]
    got = torch.compile(lambda x: mg._join_linears(x, linears), backend="aot_eager")(x)
    want = torch.cat([m(x) for m in linears], -1)
    g = torch.randn_like(want)
    for a, b in zip([got, *torch.autograd.grad(got, leaves, g)],
                    [want, *torch.autograd.grad(want, leaves, g)]):
        torch.testing.assert_close(a, b, **({} if dtype == torch.float32 else
                                            dict(rtol=2.0**-6, atol=2.0**-6)))


@pytest.mark.gpu
@pytest.mark.parametrize("build", [lambda: MinGRU(64, 64), lambda: GivensMinGRU(64, 64),
                                   lambda: DeltaMinGRU(64, 64, n_heads=2)])
def test_joined_layers_compile(cuda, build, monkeypatch):
    """A compiled fp32 layer equals the eager one."""
    monkeypatch.setenv("MINGRU_SCAN", "hip")
    print("[gpu] compiled joined layer", flush=True)
    torch.manual_seed(6)
    m = build().to(cuda)
    x = torch.randn(2, 200, 64, device=cuda, requires_grad=True)
    torch._dynamo.reset()
    y, want = torch.compile(m, backend="aot_eager")(x), m(x)
    g = torch.randn_like(want)
    leaves = [x, *m.parameters()]
    for a, b in zip([y, *torch.autograd.grad(y, leaves, g)],
                    [want, *torch.autograd.grad(want, leaves, g)]):
        assert _off(a, b) <= 2e-5


def test_joined_linears_under_transforms():
    """Forward mode and vmap, which take no Python function, take the plain product."""
    torch.manual_seed(3)
    linears = [nn.Linear(6, n) for n in (66, 2)]
    x, t = torch.randn(2, 4, 6), torch.randn(2, 4, 6)

    def separate(x):
        return torch.cat([m(x) for m in linears], -1)

    got = torch.func.jvp(lambda x: mg._join_linears(x, linears), (x,), (t,))
    torch.testing.assert_close(got, torch.func.jvp(separate, (x,), (t,)))
    torch.testing.assert_close(torch.func.vmap(lambda x: mg._join_linears(x, linears))(x), separate(x))
    torch.testing.assert_close(torch.func.grad(lambda x: mg._join_linears(x, linears).sum())(x),
                               torch.func.grad(lambda x: separate(x).sum())(x))
