"""GPU parity of the elementwise scans on bf16 tensors, read and written as bf16.

Reference: the recurrence in float64 on the bf16 inputs, differentiated by torch
autograd.  The kernels compute in fp32 and round each output once, so an output x may
be off by bf16's unit roundoff 2^-8 |x| plus the fp32 kernels' own bars (1e-4 forward,
1e-3 gradients); a recorded fp32 state that had been rounded to bf16 would exceed it.
"""

import pytest
import torch

from mingru_amd import hip_scans, linear_scan, parallel_scan_log

pytestmark = pytest.mark.gpu

ROUND = 2.0**-8
FWD_TOL, GRAD_TOL = 1e-4, 1e-3

# B, T, D: 1, 2 and 4 columns per lane; a wave's 8 steps and a chunk's 64 steps with
# remainders; one-launch aggregate and look-back forms; odd and 2-byte aligned rows.
SHAPES = [(3, 1, 64), (1, 300, 7), (2, 65, 129), (2, 777, 136), (32, 1024, 128), (2, 2113, 64),
          (8, 2048, 512), (5, 3001, 260)]


def _bf16(*shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (scale * torch.randn(*shape, generator=g)).to(torch.bfloat16)


def _scan(a, b, h):
    out = []
    for at, bt in zip(a.unbind(1), b.unbind(1)):
        h = at * h + bt
        out.append(h)
    return torch.stack(out, 1)


def _check(name, x, ref, tol):
    assert x.dtype == torch.bfloat16 and x.shape == ref.shape, name
    off = (x.double().cpu() - ref).abs() - ROUND * ref.abs()
    assert off.max().item() <= tol, f"{name}: {off.max().item():.3e} past the bf16 rounding"


def _run(cuda, fn, ref_fn, ins, gouts, names):
    leaves = [t.to(cuda).requires_grad_() for t in ins]
    refs = [t.double().requires_grad_() for t in ins]
    outs, routs = fn(*leaves), ref_fn(*refs)
    grads = torch.autograd.grad(outs, leaves, [g.to(cuda) for g in gouts])
    rgrads = torch.autograd.grad(routs, refs, [g.double() for g in gouts])
    torch.cuda.synchronize()
    for i, (x, r) in enumerate(zip(outs, routs)):
        _check(f"out{i}", x.detach(), r.detach(), FWD_TOL)
    for n, x, r in zip(names, grads, rgrads):
        _check("d" + n, x, r, GRAD_TOL * max(1.0, r.abs().max().item() / 16))
    return outs


@pytest.mark.parametrize("shape", SHAPES)
def test_linear_scan_bf16(cuda, shape):
    print(f"[gpu] linear_scan bf16 {shape}", flush=True)
    a = torch.tanh(2 * _bf16(*shape, seed=1).float()).to(torch.bfloat16)
    b, gA, gB = (_bf16(*shape, seed=s) for s in (2, 3, 4))

    def ref(a, b):
        one = torch.ones_like(a[:, 0])
        return _scan(a, torch.zeros_like(a), one), _scan(a, b, torch.zeros_like(one))

    _run(cuda, linear_scan, ref, (a, b), (gA, gB), ("a", "b"))


@pytest.mark.parametrize("shape", SHAPES)
def test_parallel_scan_log_bf16(cuda, shape):
    print(f"[gpu] parallel_scan_log bf16 {shape}", flush=True)
    B, T, D = shape
    lc = torch.nn.functional.logsigmoid(_bf16(B, T, D, seed=5))
    lv = torch.nn.functional.logsigmoid(_bf16(B, T + 1, D, seed=6))
    gh = _bf16(B, T, D, seed=7)
    _run(cuda, lambda c, v: (parallel_scan_log(c, v),),
         lambda c, v: (_scan(c.exp(), v[:, 1:].exp(), v[:, 0].exp()),), (lc, lv), (gh,),
         ("lc", "lv"))


@pytest.mark.parametrize("h0_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["signed", "signed_coupled", "mingru"])
@pytest.mark.parametrize("shape", SHAPES)
def test_gate_scans_bf16(cuda, shape, kind, h0_dtype):
    print(f"[gpu] gate scan bf16 {kind} {shape} h0 {h0_dtype}", flush=True)
    B, T, D = shape
    s, z, hp, gh = (_bf16(B, T, D, seed=8 + i) for i in range(4))
    h0 = _bf16(B, 1, D, seed=12).to(h0_dtype)
    if kind == "mingru":
        def fn(s, hp, h0):
            return (hip_scans.mingru_gate_scan_impl(s, hp, h0),)

        def ref(k, hp, h0):
            g = torch.where(hp >= 0, hp + 0.5, torch.sigmoid(hp))
            return (_scan(torch.sigmoid(-k), torch.sigmoid(k) * g, h0[:, 0].exp()),)

        ins, names = (s, hp, h0), ("k", "hpre", "log_h0")
    else:
        def fn(s, z, hp, h0):
            return (hip_scans.signed_gate_scan_impl(s, z, hp, h0,
                                                    coupled=kind == "signed_coupled"),)

        def ref(s, z, hp, h0):
            sg, a = torch.sigmoid(z), torch.tanh(s)
            a = (1 - sg) * a if kind == "signed_coupled" else a
            return (_scan(a, sg * hp, h0[:, 0]),)

        ins, names = (s, z, hp, h0), ("s", "z", "hpre", "h0")
    if h0_dtype == torch.float32:
        ins = (*ins[:-1], h0.detach())  # its gradient comes back in fp32: checked as bf16-rounded
        names = names[:-1]
        fixed = ins[-1]
        _run(cuda, lambda *t: fn(*t, fixed.to(cuda)), lambda *t: ref(*t, fixed.double()),
             ins[:-1], (gh,), names)
    else:
        _run(cuda, fn, ref, ins, (gh,), names)


@pytest.mark.parametrize("shape", [(2, 777, 136), (3, 300, 70), (2, 3000, 512)])
@pytest.mark.parametrize("kind", ["signed", "mingru"])
def test_gate_scans_bf16_decay(cuda, shape, kind):
    """Decay in fp32 on bf16 pre-activations: its gradients stay fp32."""
    print(f"[gpu] gate scan bf16 decay {kind} {shape}", flush=True)
    B, T, D = shape
    s, z, hp, gh = (_bf16(B, T, D, seed=20 + i) for i in range(4))
    h0 = _bf16(B, 1, D, seed=24)
    g = torch.Generator().manual_seed(25)
    dt, lam = 2 * torch.rand(B, T, generator=g), 0.1 + torch.rand(D, generator=g)
    pre = (s, hp) if kind == "mingru" else (s, z, hp)
    leaves = [t.to(cuda).requires_grad_() for t in (*pre, h0, dt, lam)]
    refs = [t.double().requires_grad_() for t in (*pre, h0, dt, lam)]
    gam = torch.exp(-refs[-1] * refs[-2].unsqueeze(-1))
    if kind == "mingru":
        h = hip_scans.mingru_gate_scan_impl(*leaves)
        k, u = refs[:2]
        gg = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
        hr = _scan(torch.sigmoid(-k) * gam, torch.sigmoid(k) * gg, refs[2][:, 0].exp())
    else:
        h = hip_scans.signed_gate_scan_impl(*leaves[:4], coupled=False, dt=leaves[4],
                                            lam=leaves[5])
        hr = _scan(torch.tanh(refs[0]) * gam, torch.sigmoid(refs[1]) * refs[2], refs[3][:, 0])
    grads = torch.autograd.grad(h, leaves, gh.to(cuda))
    rgrads = torch.autograd.grad(hr, refs, gh.double())
    torch.cuda.synchronize()
    _check("h", h.detach(), hr.detach(), FWD_TOL)
    for x, r in zip(grads[:-2], rgrads[:-2]):
        _check("grad", x, r, GRAD_TOL * max(1.0, r.abs().max().item() / 16))
    for x, r in zip(grads[-2:], rgrads[-2:]):
        assert x.dtype == torch.float32
        assert (x.double().cpu() - r).abs().max().item() <= GRAD_TOL * max(1.0, r.abs().max().item())
