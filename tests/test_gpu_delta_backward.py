"""GPU parity of the delta-rule prefill backward (prime_delta_prefill_backward)
against fp64 torch autograd of the restatement in tests/delta_ref.py (the
autograd graph of chunked_delta_prime.py:73-87, 177-283; the restatement is
pinned to the C oracle and its autograd to central differences in
tests/test_oracle.py), on the CPU with the same (bf16-rounded where bf16)
inputs.  Gradients in q, k, v, beta, alpha and the incoming state, with
dy and a gradient on the final state, ragged L, the per-chunk clamp engaged or
not, grouped k/v heads; the module's autograd through it.  The one-token step
(prime_delta_decode_step_backward) likewise, against the step restatement."""
import pytest
import torch

import delta_ref as R
from prime_moment_attention import _lib

from gpu_util import dev

pytestmark = pytest.mark.gpu

TOL = 1e-3  # max|d| / max|ref| per gradient: the backward is fp32 arithmetic throughout


def _rel(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return float((a - b).abs().max() / b.abs().max().clamp_min(1e-30))


def _case(B, H, Hkv, L, seed, dtype):
    g = torch.Generator().manual_seed(seed)
    D = 64
    q = torch.nn.functional.normalize(torch.randn(B, H, L, D, generator=g), dim=-1) / 8
    k = torch.nn.functional.normalize(torch.randn(B, Hkv, L, D, generator=g), dim=-1)
    v = torch.randn(B, Hkv, L, D, generator=g)
    q, k, v = (t.to(dtype).float() for t in (q, k, v))  # the values both sides see
    beta = torch.sigmoid(torch.randn(B, H, L, generator=g)) * 0.5
    alpha = 0.9995 * (1 - 0.5 * torch.sigmoid(torch.randn(B, H, L, generator=g) - 2.5))
    s0 = torch.randn(B, H, D, 2 * D, generator=g) * 0.2
    dy = torch.randn(B, H, L, D, generator=g)
    ds = torch.randn(B, H, D, 2 * D, generator=g) * 0.1
    return q, k, v, beta, alpha, s0, dy, ds


def _reference(q, k, v, beta, alpha, s0, dy, ds, bound):
    """fp64 autograd of the restatement; grouped k/v heads expanded by repeat."""
    H, Hkv = q.shape[1], k.shape[1]
    xs = [t.double().clone().requires_grad_(True) for t in (q, k, v, beta, alpha, s0)]
    kk = xs[1].repeat_interleave(H // Hkv, 1)
    vv = xs[2].repeat_interleave(H // Hkv, 1)
    y, S = R.delta_chunked(xs[0], kk, vv, xs[3], xs[4], 0.9995, 1e-5, bound, 64, xs[5])
    loss = (y * dy.double()).sum() + (S * ds.double()).sum()
    return torch.autograd.grad(loss, xs)


@pytest.mark.parametrize("B,H,Hkv,L,bound,dtype", [
    (2, 2, 2, 64 * 3 + 17, 25.0, torch.float32),
    (1, 2, 2, 64 * 2 + 5, 2.0, torch.float32),    # the clamp engaged in some chunks
    (1, 4, 2, 100, 25.0, torch.bfloat16),         # grouped k/v heads, bf16 inputs
    (1, 2, 2, 2048, 3.0, torch.bfloat16),         # 32 chunks, clamp engaged
    (1, 1, 1, 1, 25.0, torch.float32),            # one token
])
def test_delta_backward_matches_fp64_autograd(B, H, Hkv, L, bound, dtype):
    q, k, v, beta, alpha, s0, dy, ds = _case(B, H, Hkv, L, L + H, dtype)
    print(f"[delta bwd] B={B} H={H} Hkv={Hkv} L={L} bound={bound} {dtype}", flush=True)
    to = lambda t, dt=torch.float32: t.to(dev(), dt).contiguous()
    got = _lib.delta_prefill_backward(to(q, dtype), to(k, dtype), to(v, dtype), to(beta), to(alpha), 0.9995, 1e-5,
                                      bound, to(s0), to(dy, dtype), to(ds))
    torch.cuda.synchronize()
    ref = _reference(q, k, v, beta, alpha, s0, dy.to(dtype).float(), ds, bound)
    for name, g, r in zip(("q", "k", "v", "beta", "alpha", "state"), got, ref):
        assert torch.isfinite(g).all(), name
        assert _rel(g, r) < TOL, (name, _rel(g, r))


@pytest.mark.parametrize("L,bound", [(63, 25.0), (64, 0.0), (65, 1.0), (128, 25.0), (191, 1.0), (321, 1.5)])
def test_delta_backward_chunk_edges(L, bound):
    """One to six chunks (the chains take chunks in pairs), lengths around a
    chunk's end, no clamp, a clamp that holds in every chunk."""
    args = _case(2, 2, 2, L, 40 + L, torch.float32)
    to = lambda t: t.to(dev()).contiguous()
    q, k, v, beta, alpha, s0, dy, ds = args
    got = _lib.delta_prefill_backward(*(to(t) for t in (q, k, v, beta, alpha)), 0.9995, 1e-5, bound, to(s0), to(dy),
                                      to(ds))
    torch.cuda.synchronize()
    ref = _reference(q, k, v, beta, alpha, s0, dy, ds, bound)
    for name, g, r in zip(("q", "k", "v", "beta", "alpha", "state"), got, ref):
        assert _rel(g, r) < 1e-5, (name, _rel(g, r))  # fp32 sums of up to 128 products a contraction


def test_delta_backward_sequence_groups():
    """More sequences than one workspace group holds: the later group's results
    equal those of a call with its sequences alone."""
    H, L = 120, 3
    B = 235  # 28200 (sequence, head) pairs, two a CU in a group
    per = _lib.delta_backward_workspace_size(1, 1, L)
    assert _lib.delta_backward_workspace_size(B, H, L) < per * B * H
    q, k, v, beta, alpha, s0, dy, ds = (t.to(dev()).contiguous() for t in _case(B, H, H, L, 9, torch.float32))
    got = _lib.delta_prefill_backward(q, k, v, beta, alpha, 0.9995, 1e-5, 2.0, s0, dy, ds)
    cut = B - 12
    for sel in (slice(0, 2), slice(cut, B)):
        part = _lib.delta_prefill_backward(*(t[sel].contiguous() for t in (q, k, v, beta, alpha)), 0.9995, 1e-5, 2.0,
                                           s0[sel].contiguous(), dy[sel].contiguous(), ds[sel].contiguous())
        torch.cuda.synchronize()
        for g, r in zip(got, part):
            assert torch.equal(g[sel], r)


def test_delta_backward_without_state_gradient_inputs():
    """No incoming state and no gradient on the final state: the adjoint starts
    at zero, dstate_in is not produced."""
    q, k, v, beta, alpha, _, dy, _ = _case(1, 2, 2, 64 + 30, 7, torch.float32)
    to = lambda t: t.to(dev()).contiguous()
    got = _lib.delta_prefill_backward(to(q), to(k), to(v), to(beta), to(alpha), 0.9995, 1e-5, 25.0, None, to(dy),
                                      None)
    torch.cuda.synchronize()
    assert got[5] is None
    xs = [t.double().clone().requires_grad_(True) for t in (q, k, v, beta, alpha)]
    y, _ = R.delta_chunked(*xs, 0.9995, 1e-5, 25.0, 64, None)
    ref = torch.autograd.grad((y * dy.double()).sum(), xs)
    for name, g, r in zip(("q", "k", "v", "beta", "alpha"), got, ref):
        assert _rel(g, r) < TOL, (name, _rel(g, r))


def test_delta_module_trains_through_the_chunked_branch():
    """ChunkedGatedDeltaPrimeAttention under autograd (the reference trains
    through this branch, chunked_delta_prime.py:177-283): gradients of every
    parameter and of the input against an fp64 CPU composition of the same
    module (torch projections, LayerNorm, gates and the restatement)."""
    from prime_moment_attention import ChunkedGatedDeltaPrimeAttention
    torch.manual_seed(3)
    hidden, H, D, L = 128, 2, 64, 150
    m = ChunkedGatedDeltaPrimeAttention(hidden, H, D, lyapunov_bound=4.0).to(dev())
    x = torch.randn(2, L, hidden, device=dev(), requires_grad=True)
    state = (torch.randn(2, H, D, 2 * D, device=dev()) * 0.1).requires_grad_(True)
    out, s = m(x, state=state, return_state=True)
    g = torch.Generator().manual_seed(4)
    ro = torch.randn(out.shape, generator=g)
    rs = torch.randn(s.shape, generator=g)
    ((out * ro.to(dev())).sum() + (s * rs.to(dev())).sum()).backward()

    mc = ChunkedGatedDeltaPrimeAttention(hidden, H, D, lyapunov_bound=4.0).double()
    mc.load_state_dict({k: v.detach().double().cpu() for k, v in m.state_dict().items()})
    xc = x.detach().double().cpu().requires_grad_(True)
    sc = state.detach().double().cpu().requires_grad_(True)
    B = 2
    q = mc.q_proj(xc).view(B, L, H, D).transpose(1, 2)
    k = mc.k_proj(xc).view(B, L, H, D).transpose(1, 2)
    v = mc.v_proj(xc).view(B, L, H, D).transpose(1, 2)
    q, k = mc.q_norm(q) * mc.scaling, mc.k_norm(k)
    bg = torch.sigmoid(mc.erase_proj(xc)).view(B, L, H, D).mean(-1).transpose(1, 2)
    wg = torch.sigmoid(mc.write_proj(xc)).view(B, L, H, D).mean(-1).transpose(1, 2)
    y, S = R.delta_chunked(q, k, v, wg * 0.5, mc.decay * (1 - bg * 0.5), mc.decay, mc.eps, 4.0, 64, sc)
    oc = mc.o_proj(y.transpose(1, 2).reshape(B, L, H * D))
    ((oc * ro.double()).sum() + (S * rs.double()).sum()).backward()
    assert _rel(out, oc) < TOL
    assert _rel(x.grad, xc.grad) < TOL and _rel(state.grad, sc.grad) < TOL
    for (name, p), (_, pc) in zip(m.named_parameters(), mc.named_parameters()):
        assert p.grad is not None, name
        assert _rel(p.grad, pc.grad) < TOL, (name, _rel(p.grad, pc.grad))


def _step_case(B, H, Hkv, D, seed, dtype, bound):
    g = torch.Generator().manual_seed(seed)
    q = torch.nn.functional.normalize(torch.randn(B, H, D, generator=g), dim=-1) / D ** 0.5
    k = torch.randn(B, Hkv, D, generator=g)
    v = torch.randn(B, Hkv, D, generator=g)
    q, k, v = (t.to(dtype).float() for t in (q, k, v))
    beta = torch.sigmoid(torch.randn(B, H, generator=g)) * 0.5
    alpha = 0.9995 * (1 - 0.5 * torch.sigmoid(torch.randn(B, H, generator=g) - 2.5))
    s0 = torch.randn(B, H, D, 2 * D, generator=g) * (0.3 if bound < 25.0 else 0.05)
    dy = torch.randn(B, H, D, generator=g)
    ds = torch.randn(B, H, D, 2 * D, generator=g) * 0.1
    return q, k, v, beta, alpha, s0, dy, ds


@pytest.mark.parametrize("B,H,Hkv,D,bound,dtype,with_state", [
    (3, 2, 2, 64, 25.0, torch.float32, True),
    (2, 2, 2, 64, 1.5, torch.float32, True),     # the clamp engaged
    (2, 4, 2, 64, 25.0, torch.bfloat16, True),   # grouped k/v heads, bf16 inputs
    (2, 2, 2, 32, 0.8, torch.float32, True),     # the reference test's head dim, clamp engaged
    (1, 3, 3, 7, 25.0, torch.float32, False),    # odd head dim, no incoming state
])
def test_delta_step_backward_matches_fp64_autograd(B, H, Hkv, D, bound, dtype, with_state):
    """prime_delta_decode_step_backward against fp64 autograd of the step
    restatement (tests/delta_ref.py::delta_step, pinned to oracle_delta_step
    and to central differences in tests/test_oracle.py): gradients in q, k, v,
    beta, alpha and the incoming state, with dy and a gradient on the new
    state."""
    q, k, v, beta, alpha, s0, dy, ds = _step_case(B, H, Hkv, D, 31 + D + H, dtype, bound)
    if not with_state:
        s0 = None
    print(f"[delta step bwd] B={B} H={H} Hkv={Hkv} D={D} bound={bound} {dtype} state={with_state}", flush=True)
    to = lambda t, dt=torch.float32: t.to(dev(), dt).contiguous() if t is not None else None
    got = _lib.delta_decode_step_backward(to(q, dtype), to(k, dtype), to(v, dtype), to(beta), to(alpha), 1e-5,
                                          bound, to(s0), to(dy, dtype), to(ds))
    torch.cuda.synchronize()
    xs = [t.double().clone().requires_grad_(True) for t in (q, k, v, beta, alpha)]
    sx = s0.double().clone().requires_grad_(True) if s0 is not None else None
    kk = xs[1].repeat_interleave(H // Hkv, 1)
    vv = xs[2].repeat_interleave(H // Hkv, 1)
    y, S = R.delta_step(xs[0], kk, vv, xs[3], xs[4], 1e-5, bound, sx)
    loss = (y * dy.to(dtype).double()).sum() + (S * ds.double()).sum()
    ref = torch.autograd.grad(loss, xs + ([sx] if sx is not None else []))
    names = ("q", "k", "v", "beta", "alpha", "state")
    for name, g, r in zip(names, got, ref):
        assert torch.isfinite(g).all(), name
        assert _rel(g, r) < TOL, (name, _rel(g, r))
    if s0 is None:
        assert got[5] is None


def test_delta_module_trains_through_the_step_branch():
    """ChunkedGatedDeltaPrimeAttention with one token under autograd (the
    reference's L == 1 branch is plain torch and differentiable,
    chunked_delta_prime.py:140-176): gradients of every parameter, of the
    input and of the incoming state against an fp64 CPU composition of the
    same module with the step restatement."""
    from prime_moment_attention import ChunkedGatedDeltaPrimeAttention
    torch.manual_seed(5)
    hidden, H, D, B = 128, 2, 64, 3
    m = ChunkedGatedDeltaPrimeAttention(hidden, H, D, lyapunov_bound=2.0).to(dev())
    x = torch.randn(B, 1, hidden, device=dev(), requires_grad=True)
    state = (torch.randn(B, H, D, 2 * D, device=dev()) * 0.1).requires_grad_(True)
    out, s = m(x, state=state, return_state=True)
    g = torch.Generator().manual_seed(6)
    ro = torch.randn(out.shape, generator=g)
    rs = torch.randn(s.shape, generator=g)
    ((out * ro.to(dev())).sum() + (s * rs.to(dev())).sum()).backward()

    mc = ChunkedGatedDeltaPrimeAttention(hidden, H, D, lyapunov_bound=2.0).double()
    mc.load_state_dict({k: v.detach().double().cpu() for k, v in m.state_dict().items()})
    xc = x.detach().double().cpu().requires_grad_(True)
    sc = state.detach().double().cpu().requires_grad_(True)
    q = mc.q_proj(xc).view(B, 1, H, D).transpose(1, 2)
    k = mc.k_proj(xc).view(B, 1, H, D).transpose(1, 2)
    v = mc.v_proj(xc).view(B, 1, H, D).transpose(1, 2)
    q, k = mc.q_norm(q) * mc.scaling, mc.k_norm(k)
    bg = torch.sigmoid(mc.erase_proj(xc)).view(B, 1, H, D).mean(-1).transpose(1, 2)
    wg = torch.sigmoid(mc.write_proj(xc)).view(B, 1, H, D).mean(-1).transpose(1, 2)
    y, S = R.delta_step(q[:, :, 0], k[:, :, 0], v[:, :, 0], (wg * 0.5)[..., 0], (mc.decay * (1 - bg * 0.5))[..., 0],
                        mc.eps, 2.0, sc)
    oc = mc.o_proj(y.reshape(B, 1, H * D))
    ((oc * ro.double()).sum() + (S * rs.double()).sum()).backward()
    assert _rel(out, oc) < TOL
    assert _rel(x.grad, xc.grad) < TOL and _rel(state.grad, sc.grad) < TOL
    for (name, p), (_, pc) in zip(m.named_parameters(), mc.named_parameters()):
        assert p.grad is not None, name
        assert _rel(p.grad, pc.grad) < TOL, (name, _rel(p.grad, pc.grad))


def test_delta_backward_states_and_gradients_on_any_word():
    """state_in, dstate_out and the fp32 outputs one, two and three words past a 16-byte
    boundary: the same gradients, and nothing outside the outputs written."""
    B, H, L, D = 1, 2, 130, 64
    q, k, v, beta, alpha, s0, dy, ds = _case(B, H, H, L, 77, torch.float32)
    t = [x.to(dev()).contiguous() for x in (q, k, v, dy)]
    ws = torch.empty(_lib.delta_backward_workspace_size(B, H, L), dtype=torch.uint8, device=dev())
    sizes = [B * H * L * D] * 3 + [B * H * L] * 2 + [B * H * D * 2 * D]
    runs = []
    for off in (0, 1, 2, 3):
        def shifted(x):
            buf = torch.zeros(x.numel() + 8, device=dev())
            buf[off:off + x.numel()] = x.reshape(-1).to(dev())
            return buf
        si, so, be, al = (shifted(x) for x in (s0, ds, beta, alpha))
        out = [torch.full((n + 8,), 7.0, device=dev()) for n in sizes]
        d = [_lib.tensor_desc(x, True) for x in t]
        p = lambda x: x.data_ptr() + 4 * off
        r = _lib.ctypes.byref
        rc = _lib.load().prime_delta_prefill_backward(
            r(d[0]), r(d[1]), r(d[2]), p(be), p(al), B, H, H, L, D, 64, 0.9995, 1e-5, 2.0, p(si), r(d[3]), p(so),
            *[p(x) for x in out], ws.data_ptr(), ws.numel(), _lib._stream(ws.device))
        assert rc == 0, _lib.last_error()
        torch.cuda.synchronize()
        for x, n in zip(out, sizes):
            assert (x[:off] == 7).all() and (x[off + n:] == 7).all()
        runs.append([x[off:off + n].clone() for x, n in zip(out, sizes)])
    for run in runs[1:]:
        for x, r0 in zip(run, runs[0]):
            assert torch.equal(x, r0)


def test_delta_backward_in_small_workspaces(monkeypatch):
    """A workspace for one, two and all but one sequence gives the bits of the full one;
    less than one sequence's is refused; a wrapper that cannot get the full size takes
    what it can."""
    B, H, L = 1, 5, 150
    q, k, v, beta, alpha, s0, dy, ds = (t.to(dev()).contiguous() for t in _case(B, H, H, L, 21, torch.float32))
    per = _lib.delta_backward_workspace_size(1, 1, L)
    assert _lib.delta_backward_workspace_size(B, H, L) == per * B * H

    def run(size=None):
        ws = None if size is None else torch.empty(size, dtype=torch.uint8, device=dev())
        out = _lib.delta_prefill_backward(q, k, v, beta, alpha, 0.9995, 1e-5, 2.0, s0, dy, ds, workspace=ws)
        torch.cuda.synchronize()
        return out
    ref = run(per * B * H)
    for size in (per, 2 * per, 4 * per, 2 * per + 100, 20 * per):
        assert all(torch.equal(x, r) for x, r in zip(run(size), ref))
    with pytest.raises(RuntimeError, match="below"):
        run(per - 1)
    sizes, empty = [], torch.empty

    def scarce(*a, **kw):
        if kw.get("dtype") is torch.uint8:
            sizes.append(a[0])
            if a[0] > 2 * per:
                raise torch.OutOfMemoryError("no memory")
        return empty(*a, **kw)
    monkeypatch.setattr(torch, "empty", scarce)
    assert all(torch.equal(x, r) for x, r in zip(run(), ref))
    assert sizes == [5 * per, 5 * per // 2, 5 * per // 4]
