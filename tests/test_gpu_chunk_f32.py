"""GPU parity of the fp32 chunk kernels (chunk_f32.hip) where they can go wrong:
head dims at the edges of the padded widths 16, 32 and 64, lengths around a
chunk's end and the one-token kernel's line, rows at any alignment and in mixed
dtypes, and decays of 0.  Against the float64 oracle; 2e-5 of each tensor's
largest value: fp32 sums of a few hundred products at 6e-8 each."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from prime_moment_attention import _lib

import test_gpu_selective_backward as SB
from selective_ref import selective_forward
from gpu_util import dev, random_state, state_to_dev, state_to_np, to_dev, to_np

pytestmark = pytest.mark.gpu
TOL = 2e-5


def _close(x, r, name):
    e = np.abs(np.asarray(x, np.float64).reshape(np.shape(r)) - r).max() / max(np.abs(r).max(), 1e-300)
    assert e < TOL, f"{name}: {e:.2e}"


def _case(B, H, L, D, seed):
    rng = np.random.default_rng(seed)
    q, k, v = O.make_inputs((B, H, L, D), seed=seed, bf16=False)
    lam = rng.uniform(0.98, 0.9999, H).astype(np.float32)
    return q, k, v, lam, rng


@pytest.mark.parametrize("D,L", [(1, 2), (15, 63), (16, 64), (17, 65), (31, 129), (32, 128), (33, 127), (63, 66)])
def test_chunk_f32_prefill_and_backward_edges(D, L):
    B, H = 2, 2
    BH = B * H
    q, k, v, lam, rng = _case(B, H, L, D, 100 + D)
    st0 = random_state(BH, D, 7)
    dy = rng.standard_normal((B, H, L, D)).astype(np.float32)
    ds = tuple(0.1 * rng.standard_normal(x.shape) for x in O.zero_state(BH, D))
    flat = [x.reshape(BH, L, D) for x in (q, k, v)]
    lam_bh = np.tile(lam.astype(np.float64), B)
    yo, so = O.chunked(*flat, lam_bh, eps=1.0, chunk=64, state=st0)
    ref = O.recurrent_vjp(*flat, lam_bh, dy.reshape(BH, L, D), eps=1.0, state=st0, dstate=ds)
    print(f"[chunk f32] D={D} L={L}", flush=True)
    tq, tk, tv, tl, tdy = (to_dev(x) for x in (q, k, v, lam, dy))
    st_in = state_to_dev(st0, B, H, D)
    y, st = torch.empty_like(tq), _lib.new_state(B, H, D, dev())
    _lib.chunked_prefill(tq, tk, tv, tl, 1.0, 64, st_in, y, st)
    g = [torch.empty_like(tq) for _ in range(3)]
    dsi = _lib.new_state(B, H, D, dev())
    _lib.chunked_prefill_backward(tq, tk, tv, tl, 1.0, st_in, tdy, state_to_dev(ds, B, H, D), *g, dsi)
    torch.cuda.synchronize()
    _close(to_np(y), yo.reshape(y.shape), "y")
    for n, x, r in zip("S0 S1 S2 K0 K1 K2".split(), state_to_np(st, BH, D), so):
        _close(x, r, n)
    for n, x, r in zip(("dq", "dk", "dv"), g, ref[:3]):
        _close(to_np(x), r, n)
    for n, x, r in zip("S0 S1 S2 K0 K1 K2".split(), state_to_np(dsi, BH, D), ref[3]):
        _close(x, r, "d" + n)


def test_chunk_f32_any_alignment_and_mixed_dtypes():
    """Rows that start on odd elements, q fp32, k bf16, v fp16, grouped heads:
    the same values as contiguous fp32 rows."""
    B, H, Hkv, L, D = 2, 4, 2, 70, 24
    g = torch.Generator().manual_seed(3)
    big = [torch.randn(B, h, L, D + 5, generator=g) * 0.3 for h in (H, Hkv, Hkv)]
    views = [t.to(dev(), dt)[..., 3:3 + D] for t, dt in zip(big, (torch.float32, torch.bfloat16, torch.float16))]
    lam = torch.full((H,), 0.99, device=dev())
    out = []
    for q, k, v in (views, [t.float().contiguous() for t in views]):
        y, st = torch.empty(B, H, L, D, device=dev()), _lib.new_state(B, H, D, dev())
        _lib.chunked_prefill(q, k, v, lam, 1.0, 64, None, y, st)
        out.append((y, *st))
    torch.cuda.synchronize()
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_chunk_f32_zero_decay():
    """A decay of 0 (and a log decay of -inf) keeps each token alone: y is v
    over the clamped score of its own key."""
    B, H, L, D = 1, 2, 70, 32
    q, k, v, _, _ = _case(B, H, L, D, 5)
    score = 1 + (q * k).sum(-1) + 0.5 * (q * q * k * k).sum(-1)
    want = v * (score / np.maximum(score, 1.0))[..., None]
    t = [to_dev(x) for x in (q, k, v)]
    y, y2 = torch.empty_like(t[0]), torch.empty_like(t[0])
    _lib.chunked_prefill(*t, torch.zeros(H, device=dev()), 1.0, 64, None, y, _lib.new_state(B, H, D, dev()))
    ninf = torch.full((B, H, L), -float("inf"), device=dev())
    _lib.selective_prefill(*t, ninf, torch.ones(H, device=dev()), 1.0, None, y2, _lib.new_state(B, H, D, dev()))
    torch.cuda.synchronize()
    _close(to_np(y), want, "y")
    _close(to_np(y2), want, "selective y")


@pytest.mark.parametrize("D", [32, 63])
def test_chunk_f32_dense_clamp_backward_scratch(D):
    """The dense clamp's correction in the workspace or, where a caller gives the
    per-token scratch alone, in the incoming state's adjoint: the same result."""
    B, H, L = 1, 2, 90
    q, k, v, lam, rng = _case(B, H, L, D, 11)
    st = state_to_dev(random_state(B * H, D, 12), B, H, D)
    t = [to_dev(x) for x in (q, k, v)]
    dy = to_dev(rng.standard_normal(q.shape).astype(np.float32))
    out = []
    small = (B * H * L * 8 + 255) // 256 * 256
    for size in (_lib.backward_workspace_size(B, H, L), small):
        g, dsi = [torch.empty_like(t[0]) for _ in range(3)], _lib.new_state(B, H, D, dev())
        _lib.chunked_prefill_backward(*t, to_dev(lam), 2.5, st, dy, None, *g, dsi, flags=1,
                                      workspace=torch.empty(size, dtype=torch.uint8, device=dev()))
        out.append((*g, *dsi))
    torch.cuda.synchronize()
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.parametrize("L", [65, 130, 64 * 9 + 1])
def test_chunk_f32_base_backward_segments(L):
    """Head dim 64 in fp32, few sequences: one segment, two, several of few chunks."""
    B, H, D = 1, 2, 64
    q, k, v, lam, rng = _case(B, H, L, D, 50 + L)
    st0 = random_state(B * H, D, 51)
    dy = rng.standard_normal(q.shape).astype(np.float32)
    ds = tuple(0.1 * rng.standard_normal(x.shape) for x in O.zero_state(B * H, D))
    ref = O.recurrent_vjp(*(x.reshape(B * H, L, D) for x in (q, k, v)), np.tile(lam.astype(np.float64), B),
                          dy.reshape(B * H, L, D), eps=1.0, state=st0, dstate=ds)
    g, dsi = [torch.empty(q.shape, device=dev()) for _ in range(3)], _lib.new_state(B, H, D, dev())
    _lib.chunked_prefill_backward(*(to_dev(x) for x in (q, k, v, lam)), 1.0, state_to_dev(st0, B, H, D), to_dev(dy),
                                  state_to_dev(ds, B, H, D), *g, dsi)
    torch.cuda.synchronize()
    for n, x, r in zip(("dq", "dk", "dv"), g, ref[:3]):
        _close(to_np(x), r, n)
    for n, x, r in zip("S0 S1 S2 K0 K1 K2".split(), state_to_np(dsi, B * H, D), ref[3]):
        _close(x, r, "d" + n)


@pytest.mark.parametrize("L,with_state", [(130, False), (64 * 5, True), (64 * 13 - 55, True)])
def test_chunk_f32_selective_backward_segments(L, with_state):
    """Few sequences: the selective backward in segments (every gradient, the decay
    sums carried over the segments), and in one where the workspace holds no slots."""
    B, H = 1, 3
    args = SB._case(B, H, L, 70 + L, with_state, with_state)
    q, k, v, ld, beta, dy, st, ds = args
    small = (B * H * L * 8 + 255) // 256 * 256 + B * H * (L + 1) * 4
    assert _lib.selective_backward_workspace_size(B, H, L) > small
    ref = SB._reference(*args, 1.0)
    for ws in (None, torch.empty(small, dtype=torch.uint8, device=dev())):
        g = [torch.empty(q.shape, device=dev()) for _ in range(3)]
        dld, dks = torch.empty(B, H, L, device=dev()), torch.empty(B, H, device=dev())
        dsi = _lib.new_state(B, H, 64, dev()) if with_state else None
        dst = lambda s: state_to_dev(s, B, H, 64) if s is not None else None
        _lib.selective_prefill_backward(*(to_dev(x) for x in (q, k, v, ld, beta)), 1.0, dst(st), to_dev(dy), dst(ds),
                                        *g, dsi, dld, dks, workspace=ws)
        torch.cuda.synchronize()
        for n, x in zip(("dq", "dk", "dv", "dlog_decay", "dk_scale"), (*g, dld, dks)):
            _close(to_np(x), ref[n], n)
        if with_state:
            for x, r in zip(dsi, ref["dstate_in"]):
                _close(to_np(x), r, "dstate")


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("share", [0.1, 0.5])
def test_chunk_f32_selective_strong_decays(D, share):
    """Tokens that decay by e^-25 (the module's Delta <= 50 at tau = 2) among mild ones:
    the mild decays keep fp32 precision though the chunk's log decays add up to
    hundreds.  2-norm error against float64; 1e-6 is some tens of fp32 roundings (with a
    single fp32 prefix sum y is 2e-6 to 6e-6 off here, the state 1e-5).  The log decays'
    adjoint is a suffix sum whose terms cancel (1e-6 to 4e-6 here): 1e-5."""
    B, H, L = 2, 2, 130
    q, k, v, _, rng = _case(B, H, L, D, 300 + D)
    ld = -rng.uniform(0.001, 0.2, (B, H, L))
    ld[rng.random((B, H, L)) < share] = -25.0
    ld, beta = ld.astype(np.float32), rng.uniform(0.6, 2.0, H).astype(np.float32)
    dy = rng.standard_normal(q.shape).astype(np.float32)
    t = [torch.from_numpy(x.astype(np.float64)).requires_grad_() for x in
         (q, k, v, ld, np.broadcast_to(beta, (B, H)).copy())]
    ref, st_ref = selective_forward(*t, 1.0)
    (ref * torch.from_numpy(dy.astype(np.float64))).sum().backward()
    d = [to_dev(x) for x in (q, k, v, ld, beta)]
    y, st = torch.empty(q.shape, device=dev()), _lib.new_state(B, H, D, dev())
    _lib.selective_prefill(*d, 1.0, None, y, st)
    g = [torch.empty(q.shape, device=dev()) for _ in range(3)]
    dld, dks = torch.empty(B, H, L, device=dev()), torch.empty(B, H, device=dev())
    _lib.selective_prefill_backward(*d, 1.0, None, to_dev(dy), None, *g, None, dld, dks)
    torch.cuda.synchronize()
    err = {}
    for n, x, r in zip(("y", "S0", "S1", "S2", "K0", "K1", "K2", "dq", "dk", "dv", "dld", "dbeta"),
                       (y, *st, *g, dld, dks), (ref, *st_ref, *(x.grad for x in t))):
        r = r.detach().numpy()
        err[n] = float(np.linalg.norm(to_np(x).astype(np.float64).reshape(r.shape) - r) / np.linalg.norm(r))
    print({n: f"{e:.1e}" for n, e in err.items()})
    assert err.pop("dld") < 1e-5 and max(err.values()) < 1e-6, err


@pytest.mark.parametrize("selective", [False, True])
@pytest.mark.parametrize("D,b", [(16, 0), (32, 37), (63, 79), (40, 64)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), 1e25])
def test_chunk_f32_unbounded_values_reach_only_tokens_that_see_them(selective, D, b, bad):
    """Head dims below 64: NaN, infinity or a value whose square overflows in one token's
    q, k, v or dy leaves every result that does not depend on that token as without it
    (the order of a tile's sum apart: the file's tolerance)."""
    B, H, L = 1, 2, 100
    q, k, v, lam, rng = _case(B, H, L, D, 17)
    dy = rng.standard_normal(q.shape).astype(np.float32)
    ld, beta = to_dev(np.log(rng.uniform(0.9, 1.0, (B, H, L))).astype(np.float32)), to_dev(np.ones(H, np.float32))

    def run(q, k, v, dy):
        t = [to_dev(x) for x in (q, k, v)]
        y, g = torch.empty_like(t[0]), [torch.empty_like(t[0]) for _ in range(3)]
        if selective:
            dld, dks = torch.empty(B, H, L, device=dev()), torch.empty(B, H, device=dev())
            _lib.selective_prefill(*t, ld, beta, 1.0, None, y, None)
            _lib.selective_prefill_backward(*t, ld, beta, 1.0, None, to_dev(dy), None, *g, None, dld, dks)
        else:
            _lib.chunked_prefill(*t, to_dev(lam), 1.0, 64, None, y, None)
            _lib.chunked_prefill_backward(*t, to_dev(lam), 1.0, None, to_dev(dy), None, *g, None)
        torch.cuda.synchronize()
        return [to_np(x) for x in (y, *g)]
    clean = run(q, k, v, dy)
    before, after = np.arange(L) < b, np.arange(L) > b
    other, none, every = before | after, np.zeros(L, bool), np.ones(L, bool)
    # tokens of y, dq, dk, dv that do not depend on token b's q, k, v, dy
    free = {"q": (other, other, after, after), "k": (before, before, none, none),
            "v": (before, before, none, every), "dy": (every, other, after, after)}
    for name, tokens in free.items():
        x = {"q": q.copy(), "k": k.copy(), "v": v.copy(), "dy": dy.copy()}
        x[name][:, :, b, D // 2] = bad
        for what, got, want, n in zip(("y", "dq", "dk", "dv"), run(**x), clean, tokens):
            if n.any():
                e = np.abs(got[:, :, n] - want[:, :, n]).max() / np.abs(want).max()
                assert e < TOL, (name, what, e)


@pytest.mark.parametrize("form", ["base", "dense state", "selective"])
def test_chunk_f32_gradient_rows_on_any_element(form):
    """Head dim 64, fp32: gradient rows off the four-element boundary (element stores)
    hold the bits of aligned ones (one store per four), and the padding between rows is
    left alone, for every gradient dtype."""
    B, H, L, D = 1, 2, 150, 64
    q, k, v, lam, rng = _case(B, H, L, D, 60)
    t = [to_dev(x) for x in (q, k, v)]
    dy = to_dev(rng.standard_normal(q.shape).astype(np.float32))
    ld = to_dev(np.log(rng.uniform(0.9, 1.0, (B, H, L))).astype(np.float32))
    st = state_to_dev(random_state(B * H, D, 61), B, H, D) if form == "dense state" else None

    def run(dtype, pitch):
        buf = [torch.full((B, H, L, pitch), 7.0, device=dev(), dtype=dtype) for _ in range(3)]
        g = [b[..., pitch - D:] for b in buf]
        if form == "selective":
            dld, dks = torch.empty(B, H, L, device=dev()), torch.empty(B, H, device=dev())
            _lib.selective_prefill_backward(*t, ld, to_dev(lam), 1.0, None, dy, None, *g, None, dld, dks)
        else:
            _lib.chunked_prefill_backward(*t, to_dev(lam), 1.0, st, dy, None, *g,
                                          _lib.new_state(B, H, D, dev()) if st else None, flags=1 if st else 0)
        torch.cuda.synchronize()
        assert all((b[..., :pitch - D] == 7).all() for b in buf)
        return [x.contiguous() for x in g]
    for dtype in (torch.float32, torch.bfloat16, torch.float16):
        ref = run(dtype, D)
        for pitch in (D + 1, D + 2, D + 4):
            print(f"[chunk f32 rows] {form} {dtype} pitch {pitch}", flush=True)
            for x, r in zip(run(dtype, pitch), ref):
                assert torch.equal(x, r)


def test_chunk_f32_dense_clamp_backward_in_place_state_adjoint():
    """dstate_in on the buffers of dstate_out: the same result with the correction in the
    workspace; refused where the workspace holds the per-token scratch alone (the
    correction would replace an adjoint that is still to be read)."""
    B, H, L, D = 1, 2, 90, 32
    q, k, v, lam, rng = _case(B, H, L, D, 13)
    st = state_to_dev(random_state(B * H, D, 14), B, H, D)
    ds = [0.1 * rng.standard_normal(x.shape) for x in O.zero_state(B * H, D)]
    t, dy = [to_dev(x) for x in (q, k, v)], to_dev(rng.standard_normal(q.shape).astype(np.float32))
    small = (B * H * L * 8 + 255) // 256 * 256

    def run(inplace, size):
        g, dso = [torch.empty_like(t[0]) for _ in range(3)], state_to_dev(ds, B, H, D)
        dsi = dso if inplace else _lib.new_state(B, H, D, dev())
        _lib.chunked_prefill_backward(*t, to_dev(lam), 2.5, st, dy, dso, *g, dsi, flags=1,
                                      workspace=torch.empty(size, dtype=torch.uint8, device=dev()))
        torch.cuda.synchronize()
        return (*g, *dsi)
    full = _lib.backward_workspace_size(B, H, L)
    ref = run(False, full)
    for out in (run(True, full), run(False, small)):
        assert all(torch.equal(a, b) for a, b in zip(out, ref))
    with pytest.raises(RuntimeError, match="overlaps"):
        run(True, small)
