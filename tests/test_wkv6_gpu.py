"""Parity of the HIP wkv6 forward (through the C ABI) with the CPU oracle.

Tolerance: err = max|y - ref| / max(|ref|, rms(ref)) <= 1e-3, with ref the sequential recurrence
evaluated in float64 on the same (bf16- or fp32-rounded) inputs.
"""
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


def run(ops, r, k, v, w, u, H, dtype=torch.float32, w_dtype=torch.float32):
    dev = "cuda:0"
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(dev).to(d)
    rt, kt, vt = t(r, dtype), t(k, dtype), t(v, dtype)
    wt, ut = t(w, w_dtype), t(u, torch.float32)
    B, T, C = rt.shape
    y = ops.RUN_CUDA_RWKV6(B, T, C, H, rt, kt, vt, wt, ut)
    torch.cuda.synchronize()
    assert y.dtype == torch.float32 and tuple(y.shape) == (B, T, C)
    f = lambda x: x.float().cpu().numpy()
    return y.cpu().numpy(), f(rt), f(kt), f(vt), f(wt)


def gen(B, T, H, seed, w_mean=-0.5, w_std=0.5):
    rng = np.random.default_rng(seed)
    C = H * 64
    r, k, v = (rng.standard_normal((B, T, C), dtype=np.float32) for _ in range(3))
    w = rng.normal(w_mean, w_std, (B, T, C)).astype(np.float32)
    u = rng.normal(0.0, 0.1, (H, 64)).astype(np.float32)
    return r, k, v, w, u


def test_golden_fixtures(ops):
    for name, a in load_golden("wkv6_golden").items():
        print("case", name, flush=True)
        H = a["u"].shape[0]
        y, *_ = run(ops, a["r"], a["k"], a["v"], a["w"], a["u"], H)
        assert rel_err(y, a["y"]) <= TOL, name


@pytest.mark.parametrize("B,T,H", [(1, 1, 1), (2, 7, 2), (1, 64, 1), (2, 65, 3), (1, 196, 2), (1, 300, 1)])
def test_shapes_fp32(ops, B, T, H):
    from oracle import clib
    r, k, v, w, u = gen(B, T, H, B * 100 + T)
    y, *_ = run(ops, r, k, v, w, u, H)
    assert rel_err(y, clib.wkv6_fwd(r, k, v, w, u, H)) <= TOL


def test_config3_bf16(ops):
    """B=64, T=196, C=768, H=12, bf16 r,k,v (w fp32): against the sequential recurrence on the
    same bf16-rounded inputs."""
    from oracle import clib
    B, T, H = 64, 196, 12
    r, k, v, w, u = gen(B, T, H, 3)
    y, rr, kr, vr, wr = run(ops, r, k, v, w, u, H, torch.bfloat16)
    assert rel_err(y, clib.wkv6_fwd(rr, kr, vr, wr, u, H)) <= TOL
    y2, rr, kr, vr, wr = run(ops, r, k, v, w, u, H, torch.bfloat16, torch.bfloat16)
    assert rel_err(y2, clib.wkv6_fwd(rr, kr, vr, wr, u, H)) <= TOL


@pytest.mark.parametrize("w_mean", [-8.0, 1.5, 4.0])
def test_extreme_decay(ops, w_mean):
    """d ~ 1 (no decay), strong decay, and d == 0 (only t-1, t, t+1 contribute)."""
    from oracle import clib
    r, k, v, w, u = gen(2, 100, 2, 11, w_mean=w_mean, w_std=0.3)
    y, *_ = run(ops, r, k, v, w, u, 2)
    assert np.isfinite(y).all()
    assert rel_err(y, clib.wkv6_fwd(r, k, v, w, u, 2)) <= TOL


def test_chunked_and_sequential_kernels_agree(ops, force):
    """The matrix-core path and the sequential-state path are independent implementations."""
    r, k, v, w, u = gen(3, 196, 2, 21)
    y_chunk, *_ = run(ops, r, k, v, w, u, 2, torch.bfloat16)
    force("wkv6_fwd_scalar")
    y_seq, *_ = run(ops, r, k, v, w, u, 2, torch.bfloat16)
    assert rel_err(y_chunk, y_seq) <= TOL


def test_mixed_ranges_fall_back_per_sequence(ops):
    """One head with a decay far outside the chunked kernel's range, the other ordinary."""
    from oracle import clib
    r, k, v, w, u = gen(2, 130, 2, 31)
    w[:, :, :64] = 3.0 + 0.2 * w[:, :, :64]
    y, *_ = run(ops, r, k, v, w, u, 2)
    assert np.isfinite(y).all()
    assert rel_err(y, clib.wkv6_fwd(r, k, v, w, u, 2)) <= TOL


def test_reversal_and_head_independence(ops):
    r, k, v, w, u = gen(2, 50, 2, 5)
    y, *_ = run(ops, r, k, v, w, u, 2)
    yr, *_ = run(ops, r[:, ::-1], k[:, ::-1], v[:, ::-1], w[:, ::-1], u, 2)
    assert np.abs(yr[:, ::-1] - y).max() <= 1e-3 * np.sqrt((y ** 2).mean())
    sw = lambda a: np.concatenate([a[..., 64:], a[..., :64]], axis=-1)
    ys, *_ = run(ops, sw(r), sw(k), sw(v), sw(w), u[::-1], 2)
    assert np.abs(sw(ys) - y).max() <= 1e-3 * np.sqrt((y ** 2).mean())


def test_error_behaviour(ops):
    x = torch.randn(1, 4, 64, device="cuda")
    u = torch.zeros(1, 64, device="cuda")
    with pytest.raises(AssertionError):
        ops.RUN_CUDA_RWKV6(1, 4, 64, 2, x, x, x, x, u)           # HEAD_SIZE != C // H
    with pytest.raises(AssertionError):
        ops.RUN_CUDA_RWKV6(1, 4, 64, 1, x.transpose(1, 2).contiguous().transpose(1, 2), x, x, x, u)
    with pytest.raises(RuntimeError):
        ops.wkv6_forward(1, 4, 64, 1, x.cpu(), x, x, x, u)


@pytest.mark.parametrize("T", [200, 300])
def test_phase_stamping_entry_point(ops, T):
    """vrwkv_wkv6_fwd_phases (the chunked kernel writing a shader-clock stamp at six points of every wave's chunk
    steps, which bench.py turns into its per-phase figures): the chunked kernel's own y bit for bit, every stamp
    written, and the stamps of a wave in program order -- stage E entered, operands written, behind the barrier, matrix
    stage entered, y stored, behind the barrier -- within a step and from step to step.  Also its argument checks."""
    import ctypes
    lib = ops.lib()
    dev = "cuda:0"
    B, H = 3, 2
    C = H * 64
    r, k, v, w, u = gen(B, T, H, 77)
    tt = lambda a, d: torch.from_numpy(a).to(dev).to(d)
    rt, kt, vt, wt, ut = tt(r, torch.bfloat16), tt(k, torch.bfloat16), tt(v, torch.bfloat16), tt(w, torch.float32), tt(u, torch.float32)
    want = ops.wkv6_forward(B, T, C, H, rt, kt, vt, wt, ut, whole=True)
    nb = lib.vrwkv_wkv6_fwd_phases_bytes(B, T, H)
    nchunk = (T + 31) // 32
    assert nb == B * H * 8 * nchunk * 8 * 8
    st = torch.zeros(nb // 8, dtype=torch.int64, device=dev)
    y = torch.full((B, T, C), float("nan"), device=dev)
    stream = torch.cuda.current_stream().cuda_stream
    args = (rt.data_ptr(), kt.data_ptr(), vt.data_ptr(), wt.data_ptr(), ut.data_ptr(), y.data_ptr(), B, T, C, H)
    assert lib.vrwkv_wkv6_fwd_phases(*args, st.data_ptr(), nb, stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(y, want)
    s = st.cpu().numpy().reshape(B * H, 8, nchunk, 8)
    pts = s[..., [0, 1, 2, 4, 5, 6]]
    assert (pts > 0).all()
    assert (np.diff(pts, axis=-1) >= 0).all()                       # inside a step
    assert (s[:, :, 1:, 0] >= s[:, :, :-1, 6]).all()                # from step to step
    # a stamp buffer that is too small, or missing, is refused before anything is launched
    assert lib.vrwkv_wkv6_fwd_phases(*args, st.data_ptr(), nb - 8, stream) == 5
    assert lib.vrwkv_wkv6_fwd_phases(*args, None, nb, stream) == 1
    assert lib.vrwkv_wkv6_fwd_phases_bytes(0, T, H) == 0


@pytest.mark.parametrize("T,segments", [(33, 2), (64, 2), (65, 3), (250, 4), (250, 8), (577, 5), (2080, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_sequences_cut_into_segments(ops, T, segments, dtype):
    """Sequences handed to several workgroups (a forced number of segments: one chunk each, a last segment of one token,
    the most there are) meet the oracle like whole ones."""
    from oracle import clib
    r, k, v, w, u = gen(2, T, 2, seed=T + segments, w_mean=-3.0, w_std=1.0)
    with ops.option("wkv6_segments", segments):
        y, *inputs = run(ops, r, k, v, w, u, 2, dtype, dtype)
    assert rel_err(y, clib.wkv6_fwd(*inputs, u, 2)) <= TOL


def test_cut_sequence_with_a_decay_out_of_range(ops):
    """One of four sequences decays by more than e^-60 inside a chunk of its last segment: it is redone by the sequential
    recurrence, the others are not disturbed."""
    from oracle import clib
    r, k, v, w, u = gen(2, 200, 2, seed=7, w_mean=-3.0, w_std=1.0)
    w[1, 180:190, 64:] = 3.0
    with ops.option("wkv6_segments", 3):
        y, *inputs = run(ops, r, k, v, w, u, 2)
    assert rel_err(y, clib.wkv6_fwd(*inputs, u, 2)) <= TOL


@pytest.mark.parametrize("T,segments", [(300, 2), (577, 3), (2048, 8), (2080, 64), (2049, 17), (8300, 0)])
@pytest.mark.parametrize("w_mean", [-3.0, -0.8, 0.2])
def test_bf16_segments_of_two_parts_and_more_than_sixteen(ops, T, segments, w_mean):
    """Segments of 129 to 256 tokens (forced, and as the plan has them beyond 8192 tokens) are two parts each, more than sixteen get their states from a launch
    of its own; at 1.8 log2 a token the larger ones are out of a part's range and run the chunked kernel's code.  Against the sequential recurrence (bounds of
    test_sequences_as_one_or_two_products); r alone off 4 bytes gives the same bits."""
    H = 2
    x = [torch.from_numpy(a).cuda() for a in gen(2, T, H, seed=T, w_mean=w_mean, w_std=0.05 if w_mean > -3 else 0.5)]
    u = x.pop()
    x = [a.to(torch.bfloat16) for a in x]
    need = ops.lib().vrwkv_wkv6_fwd_workspace_bytes(2, T, 64 * H, H)
    with ops.option("wkv6_segments", segments):
        assert segments or need > 0
        y = ops.wkv6_forward(2, T, 64 * H, H, *x, u)
        x[0] = torch.empty(x[0].numel() + 1, dtype=torch.bfloat16, device="cuda")[1:].view_as(x[0]).copy_(x[0])
        off = ops.wkv6_forward(2, T, 64 * H, H, *x, u)
    with ops.option("wkv6_fwd_scalar", 1):
        ref = ops.wkv6_forward(2, T, 64 * H, H, *x, u)
    assert not torch.equal(y, ops.wkv6_forward(2, T, 64 * H, H, *x, u, whole=True))
    assert (y - ref).norm() <= 1.6e-5 * ref.norm() and torch.equal(off, y)


@pytest.mark.parametrize("T", [1, 15, 16, 17, 32, 33, 96, 127, 128, 129, 160, 161, 225, 256])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_sequences_as_one_or_two_products(ops, T, dtype):
    """Up to 256 tokens in one or two parts of 16-token tiles against the sequential recurrence (5e-7 of the norm): every operand rounded at its 18th bit
    (r~, k~, A or the state) and the tail x tail products left out, 2^-18 each, are 1.6e-5 at most.  A decay of 1.4 a token is beyond a part's range from
    about 100 tokens on (the chunked kernel's code takes over), single strong tokens are not; 16-bit rows off 4 bytes give the same bits."""
    H = 2
    for w_mean, spikes in ((-3.0, False), (0.3, False), (-3.0, True)):
        x = [torch.from_numpy(a).cuda() for a in gen(2, T, H, seed=T, w_mean=w_mean, w_std=0.3)]
        u = x.pop()
        if spikes:
            x[3][1, 5::40, 64:] = 2.3                                    # e^-10 at these tokens
        x = [a.to(dtype) for a in x]
        y = ops.wkv6_forward(2, T, 64 * H, H, *x, u)
        with ops.option("wkv6_fwd_scalar", 1):
            ref = ops.wkv6_forward(2, T, 64 * H, H, *x, u)
        assert (y - ref).norm() <= 1.6e-5 * ref.norm(), (w_mean, spikes)
        if dtype != torch.float32:
            off = [torch.empty(a.numel() + 1, dtype=dtype, device="cuda")[1:].view_as(a).copy_(a) for a in x]
            assert torch.equal(ops.wkv6_forward(2, T, 64 * H, H, *off, u), y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T", [1, 32, 129, 196, 256])
def test_what_autograd_records_in_16_bits_goes_chunk_by_chunk(ops, T, dtype):
    """A 16-bit forward that is recorded has the bits of the uncut entry at every length, through the host module and through the Python class; y is within
    the rounding of the split operands of the one that is not recorded (either 5e-6 of the norm from float64)."""
    H = 2
    x = [torch.from_numpy(a).cuda() for a in gen(2, T, H, seed=T, w_mean=-3.0, w_std=0.5)]
    u = x.pop()
    x = [a.to(dtype).requires_grad_() for a in x]
    args = (2, T, 64 * H, H, *x, u)
    with torch.no_grad():
        whole, plain = ops.wkv6_forward(*args, whole=True), ops.RUN_CUDA_RWKV6(*args)
    assert (whole - plain).norm() <= 1.6e-5 * whole.norm()
    for y in (ops.RUN_CUDA_RWKV6(*args), ops.WKV_6.apply(*args)):
        assert torch.equal(y, plain if dtype == torch.float32 else whole)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [300, 577, 1056, 1057])
def test_sequences_are_cut_where_autograd_records_nothing(ops, T, dtype):
    """Under no_grad and inference_mode the bonus being a parameter changes nothing: bit-identical to the plain entry, which cuts.
    What autograd records is whole in 16 bits up to 1056 tokens, and then the same in any batch."""
    H = 3
    assert ops.lib().vrwkv_wkv6_fwd_workspace_bytes(1, T, 64 * H, H) > 0
    r, k, v, w, u = (torch.from_numpy(x).cuda() for x in gen(1, T, H, seed=T, w_mean=-3.0, w_std=0.5))
    r, k, v, w = (x.to(dtype) for x in (r, k, v, w))
    u = torch.nn.Parameter(u)
    args = (1, T, 64 * H, H, r, k, v, w)
    cut, whole = ops.wkv6_forward(*args, u.detach()), ops.wkv6_forward(*args, u.detach(), whole=True)
    assert not torch.equal(cut, whole)
    recorded = ops.RUN_CUDA_RWKV6(*args, u)
    assert recorded.grad_fn is not None and torch.equal(recorded, whole if T <= 1056 and dtype == torch.bfloat16 else cut)
    assert torch.equal(ops.RUN_CUDA_RWKV6(*args, u.detach()), cut)               # nothing requires a gradient
    for mode in (torch.no_grad, torch.inference_mode):
        with mode():
            y = ops.RUN_CUDA_RWKV6(*args, u)
        assert torch.equal(y, cut) and not y.requires_grad


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [196, 256])
def test_results_of_a_sequence_of_up_to_256_tokens_do_not_depend_on_the_batch(ops, T, dtype):
    H, B = 2, 40
    x = [torch.from_numpy(a).cuda() for a in gen(B, T, H, seed=T, w_mean=-3.0, w_std=0.5)]
    u = x.pop()
    x = [a.to(dtype).requires_grad_() for a in x]
    y = ops.RUN_CUDA_RWKV6(B, T, 64 * H, H, *x, u)
    gy = torch.randn_like(y)
    grads = torch.autograd.grad(y, x, gy)
    for b in (0, B - 1):
        one = [a.detach()[b:b + 1].requires_grad_() for a in x]
        yb = ops.RUN_CUDA_RWKV6(1, T, 64 * H, H, *one, u)
        assert torch.equal(yb[0], y[b])
        assert all(torch.equal(p[0], q[b]) for p, q in zip(torch.autograd.grad(yb, one, gy[b:b + 1].contiguous()), grads))


@pytest.mark.parametrize("B,T,H,dtype", [(8, 577, 6, torch.float32), (8, 577, 6, torch.bfloat16), (16, 577, 6, torch.bfloat16), (10, 370, 6, torch.float16),
                                         (1, 4150, 3, torch.float16), (2, 577, 6, torch.bfloat16), (2, 300, 12, torch.float32)])
def test_the_planned_cut_is_the_whole_sequence(ops, B, T, H, dtype):
    """Sequences cut as the plan of their type has it against uncut ones: either is 5e-6 of the norm from float64 at most, so 1e-5 apart; the workspace
    that is asked for serves every type."""
    C = 64 * H
    g = torch.Generator(device="cuda").manual_seed(2)
    r, k, v = (torch.randn(B, T, C, generator=g, device="cuda").to(dtype) for _ in range(3))
    w = (torch.randn(B, T, C, generator=g, device="cuda") - 3).to(dtype)
    u = torch.randn(H, 64, generator=g, device="cuda") * 0.1
    whole = ops.wkv6_forward(B, T, C, H, r, k, v, w, u, whole=True)
    y = ops.wkv6_forward(B, T, C, H, r, k, v, w, u)
    assert not torch.equal(y, whole) and (y - whole).norm() <= 1e-5 * whole.norm()
    L = ops.lib()
    dt = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[dtype]
    need = L.vrwkv_wkv6_fwd_workspace_bytes(B, T, C, H)
    out, ws = torch.empty_like(whole), torch.empty(need, dtype=torch.uint8, device="cuda")
    args = [t.data_ptr() for t in (r, k, v, w, u, out)] + [B, T, C, H, dt, dt, 0, ws.data_ptr()]
    assert L.vrwkv_wkv6_fwd(*args, need, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, y)
