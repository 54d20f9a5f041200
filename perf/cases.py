"""Performance cases: the work a user of this package has it do on one GPU.

Each case is a dict of plain values; ``op`` names the call it makes.

* ``linear_scan``, ``log_scan``, ``affine_scan``: a training pass (forward and backward)
  of the public scan primitives, as a user's own recurrent layer calls them.
* ``angle_scan``, ``delta_scan``: a training pass of the angle-fused rotation scan and of
  the chunked delta rule on ready-made heads (``hip_scans`` entry points).
* ``mixer``: a training pass of one mixer layer, projections included: the output, the
  input's gradient and every parameter's gradient.
* ``prefill``: a ``MinGRUStack`` over a prompt without gradients: outputs and states.
* ``decode``: one streaming ``MinGRUStack.step``: outputs and states.

``exact`` evaluates the same call in float64 with plain torch loops, independently of the
package's own scans.
"""

from __future__ import annotations

import math
import os

import torch
import torch.nn.functional as F

from mingru_amd import (
    DeltaMinGRU,
    GivensMinGRU,
    MinGRU,
    MinGRUStack,
    RotationMinGRU,
    SignedMinGRU,
    hip_scans,
    linear_scan,
    matrix_affine_scan,
    parallel_scan_log,
)

DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16}

# Mixer constructors by name, in their default options except where a case says otherwise.
# The rotation mixer runs without angle snapping: the snap's rounding is a step function,
# so its outputs can't be compared across roundings.
MIXERS = {
    "log": MinGRU,
    "signed": SignedMinGRU,
    "rotation": RotationMinGRU,
    "givens": GivensMinGRU,
    "delta": DeltaMinGRU,
}
HYBRID = ("log", "signed", "delta")


def listed():
    return [
        # The largest diagonal scan of the benchmark, full precision.
        dict(name="linear-large", op="linear_scan", B=16, T=4096, D=1024, dtype="float32"),
        # The same primitive in a half-precision model, with ragged sizes.
        dict(name="linear-half", op="linear_scan", B=6, T=3001, D=776, dtype="bfloat16"),
        # The log-space scan at the benchmark's small size, where latency counts.
        dict(name="log-small", op="log_scan", B=4, T=1024, D=256, dtype="float32"),
        # 2x2 planes at the benchmark's size; 8x8 blocks with few planes (the scan grid).
        dict(name="affine-planes", op="affine_scan", B=16, T=4096, n=256, k=2, v=1, dtype="float32"),
        dict(name="affine-blocks", op="affine_scan", B=16, T=1024, n=8, k=8, v=1, dtype="float32"),
        # A signed layer with learnable time decay, trained in half precision.
        dict(name="signed-layer-half", op="mixer", mixer="signed", B=8, T=2048, d=1024,
             dtype="bfloat16", decay=True),
        # A Givens layer in its default form (k = 8, three rounds), full precision.
        dict(name="givens-layer", op="mixer", mixer="givens", B=8, T=2048, d=512,
             dtype="float32", decay=False),
        # A delta layer of ordinary size and a length that is no multiple of the chunk.
        dict(name="delta-layer", op="mixer", mixer="delta", B=8, T=1000, d=256, heads=4, nh=1,
             dtype="float32", decay=False),
        # The largest delta scan of the benchmark (half-precision heads).
        dict(name="delta-large", op="delta_scan", B=8, H=8, T=8192, d=64, nh=1, gated=False,
             dtype="bfloat16"),
        # Decay-gated DeltaProduct with two micro-steps, medium length.
        dict(name="delta-gated", op="delta_scan", B=4, H=8, T=2048, d=64, nh=2, gated=True,
             dtype="bfloat16"),
        # A hybrid half-precision stack over a batch of prompts.
        dict(name="prefill", op="prefill", mixer="hybrid", layers=4, B=4, T=1531, d=512,
             dtype="bfloat16"),
        # One streaming token for a few sequences: the smallest call.
        dict(name="decode", op="decode", mixer="hybrid", layers=4, B=8, T=1, d=256,
             dtype="float32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes log-uniform, odd widths among them, within the listed costs."""
    dtype = rng.choice(["float32", "bfloat16"])
    op = rng.choice(["linear_scan", "log_scan", "affine_scan", "angle_scan", "delta_scan",
                     "mixer", "mixer", "mixer", "prefill", "decode"])
    if op in ("linear_scan", "log_scan"):
        while True:
            B, T, D = _log_int(rng, 1, 128), _log_int(rng, 16, 8192), _log_int(rng, 32, 2048)
            D = D if rng.random() < 0.25 else -(-D // 8) * 8
            if 30_000 <= B * T * D <= 60_000_000:
                return dict(op=op, B=B, T=T, D=D, dtype=dtype)
    if op == "affine_scan":
        while True:
            k = rng.choice([2, 2, 4, 8])
            v = rng.choice([1, 1, 2, k])
            B, T, n = _log_int(rng, 1, 64), _log_int(rng, 16, 4096), _log_int(rng, 4, 256)
            if 10_000 <= B * T * n * k * (k + v) <= 60_000_000:
                return dict(op=op, B=B, T=T, n=n, k=k, v=v, dtype=dtype)
    if op == "angle_scan":
        while True:
            B, T, n = _log_int(rng, 1, 32), _log_int(rng, 32, 4096), _log_int(rng, 4, 128)
            if 2_000 <= B * T * n <= 1_000_000:
                return dict(op=op, B=B, T=T, n=n, k=8, dtype=dtype)
    if op == "delta_scan":
        while True:
            B, H, T = _log_int(rng, 1, 16), rng.choice([1, 2, 4, 8]), _log_int(rng, 64, 8192)
            d, nh, gated = rng.choice([16, 32, 48, 64]), rng.choice([1, 1, 2]), rng.random() < 0.5
            if B * H * T * nh <= (400_000 if dtype == "bfloat16" else 120_000):
                return dict(op=op, B=B, H=H, T=T, d=d, nh=nh, gated=gated, dtype=dtype)
    if op == "mixer":
        kind = rng.choice(["log", "log", "signed", "signed", "rotation", "givens", "delta", "delta"])
        while True:
            B, T, d = _log_int(rng, 1, 32), _log_int(rng, 32, 4096), 16 * _log_int(rng, 4, 64)
            if 50_000 <= B * T * d <= 20_000_000:
                break
        c = dict(op=op, mixer=kind, B=B, T=T, d=d, dtype=dtype, decay=rng.random() < 0.3)
        if kind == "givens":
            # Orthogonal transitions never forget: over a sequence, angles rounded to 16 bits
            # turn the state by an arbitrary amount, so such layers train in 32 bits.
            c["dtype"] = "float32"
        if kind == "delta":
            c["heads"] = next(h for h in (4, 8, 16) if d % h == 0 and d // h <= 64)
            c["nh"] = rng.choice([1, 1, 2])
        return c
    mixer = rng.choice(["log", "signed", "delta", "hybrid", "hybrid"])
    layers, d = rng.choice([2, 3, 4]), 64 * rng.choice([2, 4, 8, 12])
    if op == "prefill":
        while True:
            B, T = _log_int(rng, 1, 16), _log_int(rng, 64, 4096)
            if B * T * d <= 6_000_000:
                return dict(op=op, mixer=mixer, layers=layers, B=B, T=T, d=d, dtype=dtype)
    return dict(op=op, mixer=mixer, layers=layers, B=_log_int(rng, 1, 128), T=1, d=d, dtype=dtype)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


class _Draws:
    """Seeded normal and uniform tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda")

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda")


def _mixer_options(case):
    kind, opts = case["mixer"], {}
    if kind == "rotation":
        opts["snap"] = None
    if kind == "delta":
        opts.update(n_heads=case["heads"], nh=case["nh"])
    if case.get("decay"):
        opts["decay"] = "learnable"
    return opts


def _stack_names(case):
    if case["mixer"] == "hybrid":
        return [HYBRID[i % len(HYBRID)] for i in range(case["layers"])]
    return [case["mixer"]] * case["layers"]


def _stack_heads(d):
    return max(4, d // 64)


def _new_module(seed, dtype, build):
    with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
        torch.manual_seed(seed)
        with torch.device("cuda"):
            return build().to(dtype)


def _new_stack(case, seed, dtype):
    names, d = _stack_names(case), case["d"]
    kw = {"delta": {"n_heads": _stack_heads(d)}} if "delta" in names else None
    return _new_module(seed, dtype, lambda: MinGRUStack(d, d, len(names), mixer=names,
                                                        mixer_kwargs=kw)).eval()


def _stack_states(case, dtype, r):
    """Carried states of a stream, as ``step`` returns them."""
    B, d, states = case["B"], case["d"], []
    for name in _stack_names(case):
        if name == "delta":
            heads = _stack_heads(d)
            states.append((0.2 * r.normal(B, heads * (d // heads) ** 2)).to(dtype))
        else:
            h = 0.5 * r.normal(B, d)
            states.append((h.abs() if name == "log" else h).to(dtype))
    return states


def _lexicographic(k):
    """Plane tables of one rotation per round over all pairs i < j."""
    pairs = [(i, j) for i in range(k) for j in range(i + 1, k)]
    perm = torch.arange(k, dtype=torch.int32).repeat(len(pairs), 1)
    sgn, p2p = torch.zeros(len(pairs), k), torch.zeros(len(pairs), k, dtype=torch.int32)
    for r, (i, j) in enumerate(pairs):
        perm[r, i], perm[r, j] = j, i
        sgn[r, i], sgn[r, j] = -1.0, 1.0
    return perm, sgn, p2p


def _log_g(x):
    return torch.log(torch.where(x >= 0, x + 0.5, torch.sigmoid(x)))


def _data(case, seed):
    """The call's tensors by name, in the case's type."""
    r, dtype, op, B, T = _Draws(seed), DTYPES[case["dtype"]], case["op"], case["B"], case["T"]
    if op == "linear_scan":
        shape = (B, T, case["D"])
        t = dict(a=torch.tanh(2 * r.normal(*shape)), b=r.normal(*shape), gA=r.normal(*shape),
                 gB=r.normal(*shape))
    elif op == "log_scan":
        D = case["D"]
        z, x = r.normal(B, T, D), r.normal(B, T, D)
        first = _log_g(r.normal(B, 1, D))
        t = dict(lc=F.logsigmoid(-z), lv=torch.cat([first, F.logsigmoid(z) + _log_g(x)], 1),
                 gh=r.normal(B, T, D))
    elif op == "affine_scan":
        n, k, v = case["n"], case["k"], case["v"]
        # Transitions with singular values around one half: noise on a scaled rotation pair.
        A = 0.15 * r.normal(B, T, n, k, k) + torch.sigmoid(r.normal(B, T, n, 1, 1)) * 0.5 * \
            torch.eye(k, device="cuda")
        t = dict(A=A, Bm=r.normal(B, T, n, k, v), gA=r.normal(B, T, n, k, k),
                 gB=r.normal(B, T, n, k, v))
    elif op == "angle_scan":
        n, k = case["n"], case["k"]
        t = dict(theta=0.5 * r.normal(B, T, n, k * (k - 1) // 2, 1),
                 gamma=torch.sigmoid(r.normal(B, T, n)), b=r.normal(B, T, n, k),
                 h0=r.normal(B, n, k), gh=r.normal(B, T, n, k))
    elif op == "delta_scan":
        H, d, nh = case["H"], case["d"], case["nh"]
        t = dict(Q=r.normal(B, H, T, d), K=F.normalize(r.normal(B, H, T, nh, d), dim=-1),
                 V=r.normal(B, H, T, nh, d), beta=2 * torch.sigmoid(r.normal(B, H, T, nh)),
                 H0=0.2 * r.normal(B, H, d, d), gy=r.normal(B, H, T, d), gH=r.normal(B, H, d, d))
        if case["gated"]:
            t["log_gamma"] = -0.5 * r.uniform(B, H, T)
    elif op == "mixer":
        t = dict(x=r.normal(B, T, case["d"]), gy=r.normal(B, T, case["d"]))
        if case["decay"]:
            t["delta_t"] = 2 * r.uniform(B, T)
    elif op == "prefill":
        t = dict(x=r.normal(B, T, case["d"]))
    else:
        t = dict(x=r.normal(B, case["d"]))
        states = _stack_states(case, dtype, r)
        return {"x": t["x"].to(dtype), "states": states}
    out = {name: x.to(dtype) for name, x in t.items()}
    for name in ("H0", "gH", "log_gamma"):  # the delta state and its decay stay in 32 bits
        if name in t:
            out[name] = t[name]
    return out


# What autograd differentiates, by op.
_GRADS = {
    "linear_scan": ("a", "b"),
    "log_scan": ("lc", "lv"),
    "affine_scan": ("A", "Bm"),
    "angle_scan": ("theta", "gamma", "b", "h0"),
    "delta_scan": ("Q", "K", "V", "beta", "H0", "log_gamma"),
    "mixer": ("x",),
}


def prepare(case, seed):
    s = {"op": case["op"], "case": case, "t": _data(case, seed)}
    dtype = DTYPES[case["dtype"]]
    s["leaves"] = [s["t"][n].requires_grad_() for n in _GRADS.get(case["op"], ()) if n in s["t"]]
    if case["op"] == "mixer":
        d = case["d"]
        m = _new_module(seed, dtype, lambda: MIXERS[case["mixer"]](d, d, **_mixer_options(case)))
        s["module"] = m
        s["leaves"] += list(m.parameters())
    elif case["op"] in ("prefill", "decode"):
        s["module"] = _new_stack(case, seed, dtype)
    elif case["op"] == "angle_scan":
        s["tables"] = [x.cuda() for x in _lexicographic(case["k"])]
        s["scale"] = torch.ones(case["B"], case["T"], case["n"], device="cuda", dtype=dtype)
    os.environ.pop("MINGRU_SCAN", None)
    return s


def run(state):
    op, t = state["op"], state["t"]
    if op == "prefill":
        with torch.no_grad():
            return state["module"](t["x"])
    if op == "decode":
        return state["module"].step(t["x"], t["states"])
    if op == "linear_scan":
        outs, gouts = linear_scan(t["a"], t["b"]), (t["gA"], t["gB"])
    elif op == "log_scan":
        outs, gouts = (parallel_scan_log(t["lc"], t["lv"]),), (t["gh"],)
    elif op == "affine_scan":
        outs, gouts = matrix_affine_scan(t["A"], t["Bm"]), (t["gA"], t["gB"])
    elif op == "angle_scan":
        outs = (hip_scans.angle_scan_impl(t["theta"], state["scale"], t["gamma"], t["b"], t["h0"],
                                          *state["tables"], has_scale=0, has_decay=1),)
        gouts = (t["gh"],)
    elif op == "delta_scan":
        heads = (t["Q"], t["K"], t["V"], t["beta"])
        if "log_gamma" in t:
            outs = hip_scans.delta_gated_scan_impl(*heads, t["log_gamma"], t["H0"], chunk_size=64)
        else:
            outs = hip_scans.delta_scan_impl(*heads, t["H0"], chunk_size=64)
        gouts = (t["gy"], t["gH"])
    else:
        outs, gouts = (state["module"](t["x"], delta_t=t.get("delta_t")),), (t["gy"],)
    grads = torch.autograd.grad(outs, state["leaves"], gouts)
    return [*(o.detach() for o in outs), *grads]


# ---------------------------------------------------------------------------
# Cost and tolerance
# ---------------------------------------------------------------------------


def _mixer_cost(kind, tokens, d, e, heads=4, nh=1, train=True):
    """Bytes and flops of one mixer layer: projections, scan, and (``train``) backward."""
    if kind == "delta":
        dk = d // heads
        widths = [d] + [d] * (2 * nh) + [heads] * nh + [d]
        scan = 8 * tokens * nh * heads * dk * dk  # the recurrence's multiply-adds
    else:
        widths = {"log": [d, d], "signed": [d, d, d], "rotation": [d, d, d // 2, d // 2],
                  "givens": [d * 3 // 2, d, d]}[kind]
        scan = {"log": 10, "signed": 12, "rotation": 20, "givens": 40}[kind] * tokens * d
    flops = 2 * tokens * d * sum(widths) + scan
    bytes_ = e * (2 * tokens * d + d * sum(widths))
    return (2 * bytes_, 3 * flops) if train else (bytes_, flops)


def work(case):
    """What one pass can't do without: each input read once, each output written once."""
    op, B, T, e = case["op"], case["B"], case["T"], 2 if case["dtype"] == "bfloat16" else 4
    if op == "linear_scan":
        n = B * T * case["D"]
        return {"bytes": 10 * e * n, "flops": 14 * n}
    if op == "log_scan":
        n = B * T * case["D"]
        return {"bytes": 8 * e * n, "flops": 40 * n}
    if op == "affine_scan":
        p, k, v = B * T * case["n"], case["k"], case["v"]
        return {"bytes": 5 * e * p * k * (k + v), "flops": 6 * p * k * k * (k + v)}
    if op == "angle_scan":
        p, k = B * T * case["n"], case["k"]
        angles = k * (k - 1) // 2
        return {"bytes": e * p * (2 * (angles + 1 + k) + angles + 1 + 3 * k),
                "flops": p * angles * (3 * 6 + 60)}
    if op == "delta_scan":
        d, nh, heads = case["d"], case["nh"], B * case["H"]
        tok = heads * T
        return {"bytes": 2 * e * tok * (d + 2 * nh * d + nh) + 3 * e * tok * d + 16 * heads * d * d,
                "flops": 3 * 8 * tok * nh * d * d}
    if op == "mixer":
        b, f = _mixer_cost(case["mixer"], B * T, case["d"], e, case.get("heads", 4),
                           case.get("nh", 1))
        return {"bytes": b, "flops": f}
    d, tokens, total = case["d"], B * T, [0, 0]
    for name in _stack_names(case):
        b, f = _mixer_cost(name, tokens, d, e, _stack_heads(d), 1, train=False)
        total[0] += e * 8 * d * d  # the MLP's weights
        total[1] += f + 16 * tokens * d * d
        total[0] += b - 2 * e * tokens * d
    states = sum(2 * e * B * (d * d // _stack_heads(d) if n == "delta" else d)
                 for n in _stack_names(case))
    return {"bytes": total[0] + 2 * e * tokens * d + states, "flops": total[1]}


def tolerance(case):
    """About four times the error seen against ``exact``, worst output of each case."""
    op = case["op"]
    if case["dtype"] == "bfloat16":
        if op in ("prefill", "decode"):
            return {"rel": 3e-2}  # roundings of one layer travel through the next ones
        return {"rel": 1.5e-2 if op == "mixer" else 7e-3}
    if op == "mixer":
        # Givens: unit-modulus transitions carry every token's rounding to the end.
        return {"rel": 5e-5 if case["mixer"] == "givens" else 1e-5, "max": 1e-2}
    if op in ("prefill", "decode"):
        return {"rel": 2e-5, "max": 1e-2}
    return {"rel": 1e-5 if op == "delta_scan" else 2e-6, "max": 1e-3}


# ---------------------------------------------------------------------------
# float64 evaluation
# ---------------------------------------------------------------------------


def _scan64(a, b, h):
    """h_t = a_t h_{t-1} + b_t over axis 1."""
    out = []
    for at, bt in zip(a.unbind(1), b.unbind(1)):
        h = at * h + bt
        out.append(h)
    return torch.stack(out, 1)


def _matrix_scan64(M, b, h):
    """h_t = M_t h_{t-1} + b_t over axis 1, (B, T, n, k, k) and (B, T, n, k, v)."""
    out = []
    for Mt, bt in zip(M.unbind(1), b.unbind(1)):
        h = Mt @ h + bt
        out.append(h)
    return torch.stack(out, 1)


def _rotations64(theta, planes, k):
    """Product of plane rotations (last leftmost), rows held apart: (..., k, k).
    ``planes``: (angle index, i, j) in application order, over theta's last axis."""
    c, s = torch.cos(theta), torch.sin(theta)
    eye = torch.eye(k, dtype=theta.dtype, device=theta.device)
    rows = [eye[i].expand(*theta.shape[:-1], k) for i in range(k)]
    for m, i, j in planes:
        cm, sm = c[..., m, None], s[..., m, None]
        rows[i], rows[j] = cm * rows[i] - sm * rows[j], sm * rows[i] + cm * rows[j]
    return torch.stack(rows, -2)


def _delta64(Q, K, V, beta, log_gamma, H):
    """The delta rule in chunks of 64 tokens: (B, H, T, ..) heads; returns y and the state."""
    T, nh = Q.shape[2], K.shape[3]
    ys = []
    for s in range(0, T, 64):
        e = min(s + 64, T)
        m = (e - s) * nh
        k, v = K[:, :, s:e].flatten(2, 3), V[:, :, s:e].flatten(2, 3)
        b, q = beta[:, :, s:e].flatten(2, 3), Q[:, :, s:e]
        cum = torch.cumsum(log_gamma[:, :, s:e], -1)
        cm = cum.repeat_interleave(nh, -1)
        order = torch.arange(m, device=q.device)
        below = order[:, None] > order[None, :]
        span = torch.exp((cm[..., :, None] - cm[..., None, :]).masked_fill(~below, 0.0))
        L = (k @ k.transpose(-1, -2)) * b[..., None, :] * span * below
        eye = torch.eye(m, dtype=q.dtype, device=q.device)
        rhs = v - torch.exp(cm)[..., None] * (k @ H)
        U = torch.linalg.solve_triangular(eye + L, rhs, upper=False, unitriangular=True)
        seen = torch.arange(e - s, device=q.device)[:, None] >= (order // nh)[None, :]
        reach = torch.exp((cum[..., :, None] - cm[..., None, :]).masked_fill(~seen, 0.0)) * seen
        y = torch.exp(cum)[..., None] * (q @ H) + ((q @ k.transpose(-1, -2)) * b[..., None, :]
                                                   * reach) @ U
        tail = torch.exp(cum[..., -1:] - cm) * b
        H = torch.exp(cum[..., -1])[..., None, None] * H + (k * tail[..., None]).transpose(-1, -2) @ U
        ys.append(y)
    return torch.cat(ys, 2), H


def _mixer64(kind, p, x, state, delta_t=None, options=None):
    """One mixer over (B, T, d) from parameters ``p`` by name; ``state`` None or as ``step``
    takes it.  Returns the outputs and the last state."""
    B, T, _ = x.shape
    o = options or {}

    def lin(name):
        return F.linear(x, p[name + ".weight"], p[name + ".bias"])

    gamma_log = None
    if delta_t is not None:
        gamma_log = -F.softplus(p["rho"]) * delta_t[..., None]
    if kind == "log":
        k, u = lin("linear_z"), lin("linear_h")
        a, b = torch.sigmoid(-k), torch.sigmoid(k) * torch.exp(_log_g(u))
        h = torch.full_like(a[:, 0], 0.5) if state is None else state
    elif kind == "signed":
        z = torch.sigmoid(lin("linear_z"))
        a, b = torch.tanh(lin("linear_s")), z * lin("linear_h")
        h = torch.zeros_like(a[:, 0]) if state is None else state
    if kind in ("log", "signed"):
        hs = _scan64(a if gamma_log is None else a * torch.exp(gamma_log), b, h)
        return hs, hs[:, -1]
    if kind in ("rotation", "givens"):
        k = 2 if kind == "rotation" else 8
        n = p["linear_z.weight"].shape[0] // k
        rounds = 1 if kind == "rotation" else 3
        half = k // 2
        planes = [(r * half + m, (r % 2 + 2 * m) % k, (r % 2 + 2 * m + 1) % k)
                  for r in range(rounds) for m in range(half)]
        M = _rotations64(lin("linear_theta").view(B, T, n, rounds * half), planes, k)
        if kind == "rotation":
            scale = torch.tanh(lin("linear_u"))
            M = M * torch.stack([torch.ones_like(scale), scale], -1)[..., None, :]
        if gamma_log is not None:
            M = M * torch.exp(gamma_log)[..., None, None]
        b = (torch.sigmoid(lin("linear_z")) * lin("linear_h")).view(B, T, n, k, 1)
        h = (p["h0"].expand(B, 1, n * k) if state is None else state).reshape(B, n, k, 1)
        hs = _matrix_scan64(M, b, h).reshape(B, T, n * k)
        return hs, hs[:, -1]
    heads, nh = o["n_heads"], o.get("nh", 1)
    dk = p["linear_q.weight"].shape[0] // heads

    def split(y):
        return y.view(B, T, heads, -1).transpose(1, 2)

    Q = split(lin("linear_q"))
    K = torch.stack([F.normalize(split(lin(f"linear_k.{j}")), dim=-1) for j in range(nh)], 3)
    V = torch.stack([split(lin(f"linear_v.{j}")) for j in range(nh)], 3)
    beta = torch.stack([2 * torch.sigmoid(split(lin(f"linear_beta.{j}"))[..., 0])
                        for j in range(nh)], 3)
    lg = torch.zeros(B, heads, T, dtype=x.dtype, device=x.device)
    if gamma_log is not None:
        lg = gamma_log.transpose(1, 2)
    H = torch.zeros(B, heads, dk, dk, dtype=x.dtype, device=x.device) if state is None else \
        state.reshape(B, heads, dk, dk)
    y, H = _delta64(Q, K, V, beta, lg, H)
    y = y.transpose(1, 2).reshape(B, T, heads * dk)
    return F.linear(y, p["out_proj.weight"], p["out_proj.bias"]), H


def _stack64(case, p, x, states):
    """A ``MinGRUStack`` over (B, T, d): outputs and the mixers' last states."""
    d, new = case["d"], []

    def norm(v, name):
        return F.layer_norm(v, (d,), p[name + ".weight"], p[name + ".bias"])

    for i, name in enumerate(_stack_names(case)):
        pre = f"blocks.{i}."
        mp = {k[len(pre) + 7:]: v for k, v in p.items() if k.startswith(pre + "mingru.")}
        h, last = _mixer64(name, mp, norm(x, pre + "norm1"), states[i],
                           options={"n_heads": _stack_heads(d)})
        new.append(last)
        x = x + h
        y = F.linear(norm(x, pre + "norm2"), p[pre + "mlp.0.weight"], p[pre + "mlp.0.bias"])
        x = x + F.linear(F.gelu(y), p[pre + "mlp.3.weight"], p[pre + "mlp.3.bias"])
    return norm(x, "norm_out"), new


def exact(case, seed):
    s = prepare(case, seed)
    op = case["op"]
    if op in ("prefill", "decode"):
        p = {k: v.detach().double() for k, v in s["module"].named_parameters()}
        x = s["t"]["x"].double()
        B = case["B"]
        if op == "decode":
            y, new = _stack64(case, p, x[:, None], [h.double() for h in s["t"]["states"]])
            return y[:, 0], [h.reshape(B, -1) for h in new]
        y, new = _stack64(case, p, x, [None] * case["layers"])
        return y, [h.reshape(B, 1, -1) for h in new]
    t = {k: v.detach().double().requires_grad_() for k, v in s["t"].items()}
    leaves = [t[n] for n in _GRADS[op] if n in t]
    if op == "linear_scan":
        one, zero = torch.ones_like(t["a"][:, 0]), torch.zeros_like(t["a"][:, 0])
        outs = (_scan64(t["a"], torch.zeros_like(t["a"]), one), _scan64(t["a"], t["b"], zero))
        gouts = (t["gA"], t["gB"])
    elif op == "log_scan":
        outs = (_scan64(t["lc"].exp(), t["lv"][:, 1:].exp(), t["lv"][:, 0].exp()),)
        gouts = (t["gh"],)
    elif op == "affine_scan":
        k = case["k"]
        eye = torch.eye(k, dtype=torch.float64, device="cuda")
        zero = torch.zeros_like(t["Bm"][:, 0])
        outs = (_matrix_scan64(t["A"], torch.zeros_like(t["A"]), eye),
                _matrix_scan64(t["A"], t["Bm"], zero))
        gouts = (t["gA"], t["gB"])
    elif op == "angle_scan":
        k = case["k"]
        pairs = [(i, j) for i in range(k) for j in range(i + 1, k)]
        M = _rotations64(t["theta"][..., 0], [(r, i, j) for r, (i, j) in enumerate(pairs)], k)
        M = M * t["gamma"][..., None, None]
        outs = (_matrix_scan64(M, t["b"][..., None], t["h0"][..., None])[..., 0],)
        gouts = (t["gh"],)
    elif op == "delta_scan":
        lg = t["log_gamma"] if "log_gamma" in t else torch.zeros_like(t["Q"][..., 0])
        outs = _delta64(t["Q"], t["K"], t["V"], t["beta"], lg, t["H0"])
        gouts = (t["gy"], t["gH"])
    else:
        p = {k: v.detach().double().requires_grad_() for k, v in s["module"].named_parameters()}
        y, _ = _mixer64(case["mixer"], p, t["x"], None, t.get("delta_t"), _mixer_options(case))
        outs, gouts = (y,), (t["gy"],)
        leaves += list(p.values())
    grads = torch.autograd.grad(outs, leaves, gouts)
    return [*(o.detach() for o in outs), *grads]
