"""Parity of the HIP wkv6 backward with autograd through the float64 closed form.
Tolerance: err = max|g - ref| / max(|ref|, rms(ref)) <= 1e-3."""
import numpy as np
import pytest
import torch

from conftest import load_golden, rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-3


@pytest.fixture(scope="module")
def ops():
    import vision_rwkv_amd
    assert torch.cuda.is_available()
    return vision_rwkv_amd


def run(ops, r, k, v, w, u, gy, H, dtype=torch.float32):
    dev = "cuda:0"
    t = lambda a, d=torch.float32: torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(dev).to(d)
    rt, kt, vt = t(r, dtype), t(k, dtype), t(v, dtype)
    B, T, C = rt.shape
    out = ops.wkv6_backward(B, T, C, H, rt, kt, vt, t(w), t(u), t(gy))
    torch.cuda.synchronize()
    f = lambda x: x.float().cpu().numpy()
    return [f(x) for x in out], f(rt), f(kt), f(vt)


def test_golden_gradient_fixture(ops):
    g = load_golden("wkv6_golden")["grad_T9"]
    (gr, gk, gv, gw, gu), *_ = run(ops, g["r"], g["k"], g["v"], g["w"], g["u"], g["gy"], 1)
    for got, name in ((gr, "gr"), (gk, "gk"), (gv, "gv"), (gw, "gw"), (gu, "gu")):
        assert rel_err(got, g[name]) <= TOL, name


@pytest.mark.parametrize("B,T,H,w_mean", [(1, 1, 1, -0.5), (2, 5, 2, -0.5), (2, 40, 1, -0.5), (1, 300, 1, -3.0), (1, 30, 1, 1.0)])
def test_against_autograd_closed_form(ops, B, T, H, w_mean):
    from oracle import wkv6
    rng = np.random.default_rng(T * 7 + H)
    C = H * 64
    r, k, v, gy = (rng.standard_normal((B, T, C)).astype(np.float32) for _ in range(4))
    w = rng.normal(w_mean, 0.5, (B, T, C)).astype(np.float32)
    u = rng.normal(0, 0.1, (H, 64)).astype(np.float32)
    (gr, gk, gv, gw, gu), *_ = run(ops, r, k, v, w, u, gy, H)
    ref = wkv6.wkv6_grads_closed(r, k, v, w, u, H, gy)
    for got, want, name in zip((gr, gk, gv, gw, gu), ref, ("gr", "gk", "gv", "gw", "gu")):
        if T == 1 and name == "gw":
            assert np.abs(got).max() <= 1e-6
            continue
        assert rel_err(got, want) <= TOL, name


def test_bf16_inputs_and_autograd_function(ops):
    from oracle import wkv6
    B, T, H = 2, 33, 2
    C = H * 64
    g = torch.Generator().manual_seed(8)
    r, k, v = (torch.randn(B, T, C, generator=g).bfloat16() for _ in range(3))
    w = torch.randn(B, T, C, generator=g) * 0.5 - 0.5
    u = torch.randn(H, 64, generator=g) * 0.1
    gy = torch.randn(B, T, C, generator=g)
    leaves = [t.cuda().requires_grad_(True) for t in (r, k, v, w, u)]
    y = ops.RUN_CUDA_RWKV6(B, T, C, H, *leaves)
    y.backward(gy.cuda())
    ref = wkv6.wkv6_grads_closed(r.float().numpy(), k.float().numpy(), v.float().numpy(), w.numpy(), u.numpy(), H, gy.numpy())
    for leaf, want, tol in zip(leaves, ref, (1e-2, 1e-2, 1e-2, TOL, TOL)):   # r,k,v grads come back in bf16
        assert rel_err(leaf.grad.float().cpu().numpy(), want) <= tol
    assert tuple(leaves[4].grad.shape) == (H, 64)


def _bf16_round(a):
    return torch.from_numpy(a).bfloat16().float().numpy()


@pytest.mark.parametrize("B,T,H,w_mean", [(1, 1, 1, -0.5), (2, 2, 1, -0.5), (2, 17, 2, -0.5), (1, 33, 1, -0.5),
                                          (2, 64, 1, -1.0), (1, 100, 2, -3.0), (2, 196, 1, -0.5),
                                          (1, 40, 1, 2.5), (2, 70, 2, 0.8)])
def test_chunked_scans_bf16_against_closed_form(ops, B, T, H, w_mean):
    """bf16 r, k, v take the matrix-core scans (w_mean = 2.5: every chunk decays below e^-60, so the
    sequences are flagged and redone by the sequential sweeps; 0.8: some are).  Reference: float64
    autograd through the closed form on the rounded inputs; all five gradients come back in fp32."""
    from oracle import wkv6
    rng = np.random.default_rng(T * 11 + H)
    C = H * 64
    r, k, v = (_bf16_round(rng.standard_normal((B, T, C)).astype(np.float32)) for _ in range(3))
    gy = rng.standard_normal((B, T, C)).astype(np.float32)
    w = rng.normal(w_mean, 0.5, (B, T, C)).astype(np.float32)
    u = rng.normal(0, 0.1, (H, 64)).astype(np.float32)
    (gr, gk, gv, gw, gu), *_ = run(ops, r, k, v, w, u, gy, H, torch.bfloat16)
    ref = wkv6.wkv6_grads_closed(r, k, v, w, u, H, gy)
    for got, want, name in zip((gr, gk, gv, gw, gu), ref, ("gr", "gk", "gv", "gw", "gu")):
        assert np.isfinite(got).all(), name
        if T <= 2 and name == "gw":
            # exactly zero (no token lies between two others); for T = 2 it is the difference a - b of two
            # equal O(10) terms, each carrying the split-bf16 products' ~3e-5
            assert np.abs(got).max() <= (1e-6 if T == 1 else 1e-3)
            continue
        # heavy decay (sequential sweeps): gw has a few O(10) entries among O(0.1) ones; fp32 keeps 1e-4 of the former
        tol = 5e-3 if (name == "gw" and w_mean > 2) else TOL
        assert rel_err(got, want) <= tol, name


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("B,T,H,w_mean", [(2, 17, 2, -0.5), (1, 33, 1, -0.5), (2, 196, 1, -0.5), (1, 100, 2, -3.0), (2, 70, 2, 0.8)])
def test_chunked_scans_fp32_fp16_against_closed_form(ops, B, T, H, w_mean, dtype):
    """fp32 and fp16 r, k, v take the matrix-core scans as well (split into bf16 head + tail like the computed
    operands); reference: float64 autograd through the closed form on the inputs as the kernel sees them."""
    from oracle import wkv6
    rng = np.random.default_rng(T * 13 + H)
    C = H * 64
    r, k, v = (torch.from_numpy(rng.standard_normal((B, T, C)).astype(np.float32)).to(dtype).float().numpy() for _ in range(3))
    gy = rng.standard_normal((B, T, C)).astype(np.float32)
    w = rng.normal(w_mean, 0.5, (B, T, C)).astype(np.float32)
    u = rng.normal(0, 0.1, (H, 64)).astype(np.float32)
    (gr, gk, gv, gw, gu), *_ = run(ops, r, k, v, w, u, gy, H, dtype)
    ref = wkv6.wkv6_grads_closed(r, k, v, w, u, H, gy)
    for got, want, name in zip((gr, gk, gv, gw, gu), ref, ("gr", "gk", "gv", "gw", "gu")):
        assert np.isfinite(got).all(), name
        # gw is ld times a running difference of two sums that nearly cancel: its worst element sits a little higher
        assert rel_err(got, want) <= (2e-3 if name == "gw" else TOL), name


def test_sequential_sweeps_fp32(ops, force):
    """The sequential kernels (the fallback of flagged sequences) on their own, fp32 inputs."""
    from oracle import wkv6
    force("wkv6_bwd_scalar")
    B, T, H = 2, 50, 2
    rng = np.random.default_rng(77)
    C = H * 64
    r, k, v, gy = (rng.standard_normal((B, T, C)).astype(np.float32) for _ in range(4))
    w = rng.normal(-0.5, 0.5, (B, T, C)).astype(np.float32)
    u = rng.normal(0, 0.1, (H, 64)).astype(np.float32)
    (gr, gk, gv, gw, gu), *_ = run(ops, r, k, v, w, u, gy, H)
    ref = wkv6.wkv6_grads_closed(r, k, v, w, u, H, gy)
    for got, want, name in zip((gr, gk, gv, gw, gu), ref, ("gr", "gk", "gv", "gw", "gu")):
        assert rel_err(got, want) <= TOL, name


def test_chunked_scans_and_sequential_sweeps_full_size(ops, force):
    """VRWKV6-B shape: the matrix-core scans and the sequential sweeps (forced through the library switch), each
    against the C oracle on every output."""
    from oracle import clib
    B, T, H = 64, 196, 12
    C = H * 64
    g = torch.Generator().manual_seed(21)
    r, k, v = (torch.randn(B, T, C, generator=g).bfloat16().cuda() for _ in range(3))
    w = (torch.randn(B, T, C, generator=g) * 0.5 - 0.5).cuda()
    u = (torch.randn(H, 64, generator=g) * 0.1).cuda()
    gy = torch.randn(B, T, C, generator=g).cuda()
    got = ops.wkv6_backward(B, T, C, H, r, k, v, w, u, gy)
    force("wkv6_bwd_scalar")
    ref = ops.wkv6_backward(B, T, C, H, r, k, v, w, u, gy)
    torch.cuda.synchronize()
    f = lambda x: x.float().cpu().numpy()
    want = clib.wkv6_bwd(f(r), f(k), f(v), f(w), f(u), f(gy), H)
    # gw is a running difference of two sums that nearly cancel: its worst element over 9.6M sits higher
    for a, b, x, name in zip(got, ref, want, ("gr", "gk", "gv", "gw", "gu")):
        assert rel_err(f(a), x) <= (2e-3 if name == "gw" else TOL), name
        assert rel_err(f(b), x) <= TOL, name                 # the sequential sweeps are plain fp32 recurrences
    # float64 closed form on one (b, h) sequence
    from oracle import wkv6
    f = lambda x: x[:1, :, :64].float().cpu().numpy()
    want = wkv6.wkv6_grads_closed(f(r), f(k), f(v), f(w), u[:1].cpu().numpy(), 1, f(gy))
    for i, name in enumerate(("gr", "gk", "gv", "gw")):
        assert rel_err(got[i][:1, :, :64].cpu().numpy(), want[i]) <= TOL, name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,H,w_lo,w_hi,gw_tol", [
    (3, 577, 12, -6.0, -1.0, 6e-4),      # the range VRWKV6 initialises its decay logits in (vrwkv6.py:157-161)
    (2, 400, 4, -8.0, 0.5, 2e-3),
    (2, 577, 4, -3.0, 1.2, 5e-3), (1, 1000, 3, -3.0, 1.2, 5e-3)])
def test_uniform_decay_ranges_on_long_sequences(ops, B, T, H, w_lo, w_hi, gw_tol, dtype):
    """Forward and every gradient on sequences of 400..1000 tokens with decay logits drawn uniformly from a range,
    against the C oracle on the inputs as the kernel sees them.  y, gr, gk, gv, gu: 1e-4 of the tensor's scale, for
    every range.  gw = ld * (running difference of two sums over the rest of the sequence): the error of the running
    difference grows like sqrt(T) and is multiplied by |ld| = exp(w), so its bound depends on the range --
    6e-4 for logits in [-6, -1], 5e-3 for logits up to 1.2 (a decay of 0.036 per token)."""
    from oracle import clib
    rng = np.random.default_rng(T + H)
    C = H * 64
    r, k, v, gy = (rng.standard_normal((B, T, C), dtype=np.float32) for _ in range(4))
    k *= 0.5
    w = rng.uniform(w_lo, w_hi, (B, T, C)).astype(np.float32)
    u = (0.5 * rng.standard_normal((H, 64))).astype(np.float32)
    dev = "cuda:0"
    t = lambda a, d=torch.float32: torch.from_numpy(a).to(dev).to(d)
    rt, kt, vt, wt, ut, gt = t(r, dtype), t(k, dtype), t(v, dtype), t(w), t(u), t(gy)
    y = ops.wkv6_forward(B, T, C, H, rt, kt, vt, wt, ut)
    grads = ops.wkv6_backward(B, T, C, H, rt, kt, vt, wt, ut, gt)
    torch.cuda.synchronize()
    f = lambda x: x.float().cpu().numpy()
    err = {"y": rel_err(f(y), clib.wkv6_fwd(f(rt), f(kt), f(vt), w, u, H))}
    want = clib.wkv6_bwd(f(rt), f(kt), f(vt), w, u, gy, H)
    for name, got, ref in zip(("gr", "gk", "gv", "gw", "gu"), grads, want):
        err[name] = rel_err(f(got), ref)
    print("  " + ", ".join(f"{n} {e:.1e}" for n, e in err.items()), flush=True)
    for name, e in err.items():
        assert e <= (gw_tol if name == "gw" else 1e-4), (name, e)


@pytest.mark.parametrize("seed,B,T,H,dtype,w_dtype", [
    (1, 2, 197, 1, torch.float32, torch.float32), (2, 1, 196, 3, torch.float32, torch.float32),
    (3, 3, 3, 5, torch.bfloat16, torch.bfloat16), (4, 3, 65, 1, torch.float16, torch.float16),
    (5, 2, 300, 2, torch.bfloat16, torch.float32), (6, 2, 513, 1, torch.bfloat16, torch.bfloat16),
    (7, 3, 33, 12, torch.float32, torch.float32), (8, 1, 256, 5, torch.float16, torch.float32)])
def test_decay_regimes_mixed_over_the_heads_of_one_call(ops, seed, B, T, H, dtype, w_dtype):
    """Every (b, h) sequence of a call with a decay logit level of its own, from -8 (no decay) over the model's range
    to 2.5 and 4 (decay e^-12 and e^-55 per token: sequences handed to the sequential sweeps), inputs of scale 0.3 to
    3 and a bonus of scale 0.1 to 5; forward and every gradient against the C oracle on the inputs as the kernel sees
    them.  y, gr, gk, gv, gu: 1e-3 (they measure below 1e-4).  gw = ld * (running difference): in a head whose decay
    is so strong that the true gw all but vanishes, what is left is the rounding of the running difference times
    |ld| = e^w (12 to 55 there), up to 1e-2 in absolute terms beside heads whose gw is of order 0.2; the bound is
    5e-3 of the tensor's scale when every level is below 1, 6e-2 otherwise.  Everything must be finite."""
    from oracle import clib
    rng = np.random.default_rng(seed)
    C = H * 64
    w = np.empty((B, T, C), np.float32)
    top = -9.0
    for b in range(B):
        for h in range(H):
            level = float(rng.choice([-8, -4, -1, 0.5, 1.5, 2.5, 4.0]))
            top = max(top, level)
            w[b, :, h * 64:(h + 1) * 64] = rng.normal(level, 0.4, (T, 64))
    r, k, v, gy = (rng.standard_normal((B, T, C), dtype=np.float32) * float(rng.choice([0.3, 1, 3])) for _ in range(4))
    u = (rng.standard_normal((H, 64)) * float(rng.choice([0.1, 1, 5]))).astype(np.float32)
    dev = "cuda:0"
    t = lambda a, d: torch.from_numpy(a).to(dev).to(d)
    rt, kt, vt, wt = t(r, dtype), t(k, dtype), t(v, dtype), t(w, w_dtype)
    ut, gt = t(u, torch.float32), t(gy, torch.float32)
    y = ops.wkv6_forward(B, T, C, H, rt, kt, vt, wt, ut)
    grads = ops.wkv6_backward(B, T, C, H, rt, kt, vt, wt, ut, gt)
    torch.cuda.synchronize()
    f = lambda x: x.float().cpu().numpy()
    err = {"y": rel_err(f(y), clib.wkv6_fwd(f(rt), f(kt), f(vt), f(wt), u, H))}
    want = clib.wkv6_bwd(f(rt), f(kt), f(vt), f(wt), u, gy, H)
    for name, got, ref in zip(("gr", "gk", "gv", "gw", "gu"), grads, want):
        assert np.isfinite(f(got)).all(), name
        err[name] = rel_err(f(got), ref)
    print("  " + ", ".join(f"{n} {e:.1e}" for n, e in err.items()), flush=True)
    for name, e in err.items():
        if name == "gw":
            assert T <= 3 or e <= (5e-3 if top < 1 else 6e-2), (name, e)
        else:
            assert e <= TOL, (name, e)


@pytest.mark.parametrize("T", [1, 15, 16, 17, 32, 33, 96, 127, 128, 161, 193, 224, 225, 256])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_gradients_of_sequences_as_one_or_two_products(ops, T, dtype):
    """Against the sequential sweeps (5e-7 of the norm).  gr, gk, gv: a rounding of 2^-18 each in D, rf, kf and the state, 1.6e-5 at most.  gw sums that of up
    to T tokens, with signs that are as good as random, times its own decay.  Decays of 1.4 a token leave the range of a part, single strong tokens do not."""
    B, H = 2, 2
    C = 64 * H
    g = torch.Generator(device="cuda").manual_seed(T)
    r, k, v = (torch.randn(B, T, C, generator=g, device="cuda").to(dtype) for _ in range(3))
    gy, u = torch.randn(B, T, C, generator=g, device="cuda"), torch.randn(H, 64, generator=g, device="cuda") * 0.3
    noise = torch.randn(B, T, C, generator=g, device="cuda") * 0.3
    for w_mean, spikes in ((-3.0, False), (-1.0, False), (0.3, False), (-3.0, True)):
        w = w_mean + noise
        if spikes:
            w[1, 5::40, 64:] = 2.3
        w = w.to(dtype)
        got = ops.wkv6_backward(B, T, C, H, r, k, v, w, u, gy)
        with ops.option("wkv6_bwd_scalar", 1):
            ref = ops.wkv6_backward(B, T, C, H, r, k, v, w, u, gy)
        for x, y in zip(got[:3] + got[4:], ref[:3] + ref[4:]):
            assert (x - y).norm() <= 1.6e-5 * y.norm(), (w_mean, spikes)
        terms = w.float().exp() * ((r.float() * ref[0]).abs() + (k.float() * ref[1]).abs())
        assert (got[3] - ref[3]).norm() <= 1.6e-5 * T ** 0.5 * terms.norm(), (w_mean, spikes)
        if dtype != torch.float32:
            off = [torch.empty(a.numel() + 1, dtype=dtype, device="cuda")[1:].view_as(a).copy_(a) for a in (r, k, v, w)]
            assert all(torch.equal(x, y) for x, y in zip(ops.wkv6_backward(B, T, C, H, *off, u, gy), got))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,segments", [(300, 3), (577, 5), (1100, 9)])
def test_cut_sequences_whose_parts_are_out_of_range(ops, T, segments, dtype):
    """1.8 log2 a token: 225 over a part of 128 tokens, whose factors hold 200, 39 nats over a chunk, whose factors hold 60.  The chunked kernels' code takes
    such segments over, from the states that every workgroup folds for itself.  Bounds as above."""
    B, H = 2, 2
    C = 64 * H
    g = torch.Generator(device="cuda").manual_seed(T)
    r, k, v = (torch.randn(B, T, C, generator=g, device="cuda").to(dtype) for _ in range(3))
    gy, u = torch.randn(B, T, C, generator=g, device="cuda"), torch.randn(H, 64, generator=g, device="cuda") * 0.3
    w = torch.full((B, T, C), -3.0, device="cuda")
    w[0] = 0.2
    w = (w + 0.05 * torch.randn(B, T, C, generator=g, device="cuda")).to(dtype)
    with ops.option("wkv6_segments", segments):
        y, got = ops.wkv6_forward(B, T, C, H, r, k, v, w, u), ops.wkv6_backward(B, T, C, H, r, k, v, w, u, gy)
    with ops.option("wkv6_fwd_scalar", 1), ops.option("wkv6_bwd_scalar", 1):
        want, ref = ops.wkv6_forward(B, T, C, H, r, k, v, w, u), ops.wkv6_backward(B, T, C, H, r, k, v, w, u, gy)
    terms = w.float().exp() * ((r.float() * ref[0]).abs() + (k.float() * ref[1]).abs())
    for b in range(B):
        for x, y_ in zip((y,) + tuple(got[:3]), (want,) + tuple(ref[:3])):
            assert (x[b] - y_[b]).norm() <= 1.6e-5 * y_[b].norm()
        assert (got[3][b] - ref[3][b]).norm() <= 1.6e-5 * T ** 0.5 * terms[b].norm()
    assert (got[4] - ref[4]).norm() <= 1.6e-5 * ref[4].norm()


@pytest.mark.parametrize("T,segments", [(100, 0), (128, 0), (196, 0), (256, 0), (577, 5)])
@pytest.mark.parametrize("dtype,log2_decay,size,gy_size", [
    (torch.float32, 1.5, 1e-10, 1.), (torch.float32, 0.95, 1e-10, 1.), (torch.float32, 0.6, 1e-10, 1.), (torch.float32, 1.5, 1., 1e-12),
    (torch.float32, 0.95, 3e10, 1.), (torch.bfloat16, 0.95, 3e10, 1.), (torch.float32, 1.5, 1e6, 1e6), (torch.float16, 1.5, 8e3, 1e3), (torch.float32, 1.5, 1., 1.)])
def test_decays_over_a_part_with_rows_of_unusual_size(ops, dtype, log2_decay, size, gy_size, T, segments):
    """The factors of a part reach 2^96 at 1.5 log2 a token: products of small rows times them would leave fp32 at its lower end, those of large ones at the
    upper.  Against the sequential recurrence and sweeps with the bounds for rows of any size (see above)."""
    B, H = 2, 2
    C = 64 * H
    g = torch.Generator(device="cuda").manual_seed(T)
    r, k, v = ((torch.randn(B, T, C, generator=g, device="cuda") * size).to(dtype) for _ in range(3))
    w = np.log(log2_decay * np.log(2)) + 0.02 * torch.randn(B, T, C, generator=g, device="cuda")
    gy, u = torch.randn(B, T, C, generator=g, device="cuda") * gy_size, torch.randn(H, 64, generator=g, device="cuda") * 0.3
    with ops.option("wkv6_segments", segments):
        y, got = ops.wkv6_forward(B, T, C, H, r, k, v, w, u), ops.wkv6_backward(B, T, C, H, r, k, v, w, u, gy)
    with ops.option("wkv6_fwd_scalar", 1), ops.option("wkv6_bwd_scalar", 1):
        want, ref = ops.wkv6_forward(B, T, C, H, r, k, v, w, u), ops.wkv6_backward(B, T, C, H, r, k, v, w, u, gy)
    error = lambda a, b: (a.double() - b.double()).norm()
    for a, b in zip((y,) + tuple(got[:3]) + tuple(got[4:]), (want,) + tuple(ref[:3]) + tuple(ref[4:])):
        assert error(a, b) <= 1.6e-5 * b.double().norm()
    terms = w.double().exp() * ((r.double() * ref[0]).abs() + (k.double() * ref[1]).abs())
    assert error(got[3], ref[3]) <= 1.6e-5 * T ** 0.5 * terms.norm()


@pytest.mark.parametrize("T,segments", [(33, 2), (65, 3), (200, 3), (250, 8), (577, 5), (280, 9)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_backward_of_sequences_cut_into_segments(ops, T, segments, dtype):
    """Forced numbers of segments (one chunk each, a last segment of one token) against the uncut sequences, which the
    tests above hold to the oracle: the same sums with the states between segments formed another way, so both carry the
    split operands' 3e-5.  gw: each side within the 1e-3 that the tests above allow against the oracle, 2e-3 apart."""
    B, H = 2, 2
    g = torch.Generator().manual_seed(T)
    r, k, v = (torch.randn(B, T, 64 * H, generator=g).to(dtype).cuda() for _ in range(3))
    w = (torch.randn(B, T, 64 * H, generator=g) - 3).to(dtype).cuda()
    u, gy = (0.3 * torch.randn(H, 64, generator=g)).cuda(), torch.randn(B, T, 64 * H, generator=g).cuda()
    with ops.option("wkv6_segments", 1):
        want = ops.wkv6_backward(B, T, 64 * H, H, r, k, v, w, u, gy)
    with ops.option("wkv6_segments", segments):
        got = ops.wkv6_backward(B, T, 64 * H, H, r, k, v, w, u, gy)
        like = ops.wkv6_backward(B, T, 64 * H, H, r, k, v, w, u, gy, like_inputs=True)
    for a, b, c, name in zip(got, want, like, ("gr", "gk", "gv", "gw", "gu")):
        assert rel_err(a.cpu().numpy(), b.cpu().numpy()) <= (2e-3 if name == "gw" else 1e-4), name
        assert torch.equal(c, a.to(c.dtype)), name                       # the same sums, rounded once


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_backward_of_a_cut_sequence_with_a_decay_out_of_range(ops, dtype):
    """One of four sequences decays by more than e^-60 inside its last segment: redone by the sequential sweeps, in every
    result type; the reference is the sequential path itself, bit for bit for that sequence."""
    B, T, H = 2, 200, 2
    g = torch.Generator().manual_seed(9)
    r, k, v = (torch.randn(B, T, 64 * H, generator=g).to(dtype).cuda() for _ in range(3))
    w = torch.randn(B, T, 64 * H, generator=g) - 3
    w[1, 180:190, 64:] = 3.0
    w = w.to(dtype).cuda()
    u, gy = (0.3 * torch.randn(H, 64, generator=g)).cuda(), torch.randn(B, T, 64 * H, generator=g).cuda()
    with ops.option("wkv6_bwd_scalar", 1):
        want = ops.wkv6_backward(B, T, 64 * H, H, r, k, v, w, u, gy, like_inputs=True)
    for segments in (1, 3):
        with ops.option("wkv6_segments", segments):
            got = ops.wkv6_backward(B, T, 64 * H, H, r, k, v, w, u, gy, like_inputs=True)
        for a, b, name in zip(got[:4], want[:4], ("gr", "gk", "gv", "gw")):
            assert torch.equal(a[1, :, 64:], b[1, :, 64:]), name
            tol = 2e-3 if dtype == torch.float32 else 1e-2               # gw at the file's tolerance; bf16 results round
            assert rel_err(a.float().cpu().numpy(), b.float().cpu().numpy()) <= tol, name
        assert rel_err(got[4].cpu().numpy(), want[4].cpu().numpy()) <= 1e-4


@pytest.mark.gpu
def test_results_passed_in_are_fp32_whatever_types_are_asked_for():
    import vision_rwkv_amd as ops
    torch.manual_seed(2)
    B, T, H = 2, 65, 2
    mk = lambda: torch.randn(B, T, 64 * H, device="cuda").bfloat16()
    r, k, v, w, u, gy = mk(), mk(), mk(), mk() - 4, torch.randn(H, 64, device="cuda"), torch.randn(B, T, 64 * H, device="cuda")
    want = ops.wkv6_backward(B, T, 64 * H, H, r, k, v, w, u, gy)
    out = [torch.full_like(t, float("nan")) for t in want]
    ops.wkv6_backward(B, T, 64 * H, H, r, k, v, w, u, gy, out=out, like_inputs=True)
    assert all(torch.equal(a, b) for a, b in zip(out, want))
