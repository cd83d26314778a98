"""q_shift, the fused shift+mix kernel and the plain-PyTorch backbone."""
import contextlib

import numpy as np
import pytest
import torch

from conftest import load_golden


def test_qshift_tensor_ops_match_index_loops():
    """CPU: the boundary's q_shift (tensor slicing) against the index-loop oracle and the fixture."""
    import vision_rwkv_amd as ops
    from oracle import qshift
    g = load_golden("qshift_golden")["q"]
    y = ops.q_shift(torch.from_numpy(g["x"]), 1, 0.25, (3, 5)).numpy()
    assert np.array_equal(y, g["y"])
    for C in (22, 18, 6, 20):              # 22, 18, 6: unequal channel groups (C*gamma not an integer)
        x = np.random.default_rng(C).standard_normal((2, 20, C)).astype(np.float32)
        assert np.array_equal(ops.q_shift(torch.from_numpy(x), 1, 0.25, (4, 5)).numpy(),
                              qshift.q_shift_loops(x, 1, 0.25, (4, 5))), C


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hp,Wp,C,dtype", [(2, 3, 5, 16, torch.float32), (2, 14, 14, 192, torch.float32),
                                              (1, 7, 9, 22, torch.float32), (1, 7, 9, 20, torch.float32),
                                              (2, 24, 24, 1024, torch.bfloat16)])
def test_fused_qshift_mix_against_oracle(B, Hp, Wp, C, dtype):
    import vision_rwkv_amd as ops
    from oracle import qshift
    rng = np.random.default_rng(C)
    x = torch.from_numpy(rng.standard_normal((B, Hp * Wp, C)).astype(np.float32)).to(dtype)
    mixes = [torch.from_numpy(rng.random(C).astype(np.float32)) for _ in range(3)]
    outs = ops.q_shift_mix(x.cuda(), [m.cuda() for m in mixes], 1, 0.25, (Hp, Wp))
    xf = x.float().numpy()
    xx = qshift.q_shift_loops(xf, 1, 0.25, (Hp, Wp))
    for o, m in zip(outs, mixes):
        want = xf * m.numpy() + xx * (1 - m.numpy())
        tol = 1e-6 if dtype == torch.float32 else 2e-2
        assert np.abs(o.float().cpu().numpy() - want).max() <= tol
    if dtype == torch.float32:                      # mix = 0 returns the shifted tensor bit-exactly
        z = ops.q_shift_mix(x.cuda(), [torch.zeros(C).cuda()], 1, 0.25, (Hp, Wp))[0]
        assert np.array_equal(z.cpu().numpy(), xx)


def test_patch_embedding_gemm_equals_convolution():
    """CPU: the stem computes Conv2d(kernel = stride = patch) as one GEMM over flattened patches."""
    import vision_rwkv_amd as ops
    torch.manual_seed(0)
    net = ops.VRWKV(img_size=32, embed_dims=32, depth=1)
    img = torch.randn(2, 3, 48, 32)
    x, res = net.embed(img)
    want = net.patch_embed(img)
    assert res == (3, 2) and torch.allclose(x, want.flatten(2).transpose(1, 2), atol=1e-5)


@pytest.mark.gpu
def test_fused_qshift_multihead_with_cls_token():
    import vision_rwkv_amd as ops
    from oracle import qshift
    rng = np.random.default_rng(1)
    x = rng.standard_normal((2, 4 * 3 + 1, 128)).astype(np.float32)
    z = ops.q_shift_mix(torch.from_numpy(x).cuda(), [torch.zeros(128).cuda()], 1, 0.25, (4, 3), head_dim=64)[0]
    assert np.array_equal(z.cpu().numpy(), qshift.q_shift_multihead_loops(x, 1, 64, (4, 3), with_cls_token=True))


@pytest.mark.gpu
def test_backbone_fused_equals_eager_and_oracle_wkv():
    """A small VRWKV: fused shift+mix vs tensor-op shift; and the HIP Bi-WKV inside the block vs the
    CPU oracle evaluated on the block's own k, v."""
    import vision_rwkv_amd as ops
    from oracle import clib
    torch.manual_seed(0)
    net = ops.VRWKV(img_size=64, embed_dims=64, depth=2, post_norm=True, init_values=0.1, key_norm=True).cuda().eval()
    img = torch.randn(2, 3, 96, 64).cuda()                 # 6x4 grid: exercises the pos-embed resize
    with torch.no_grad():
        y_fused = net(img)
        for m in net.modules():
            if hasattr(m, "fused_shift"):
                m.fused_shift = False
        ops.ops.ROW_FUSE_ENABLED = False               # every element-wise step as PyTorch ops
        try:
            y_eager = net(img)
        finally:
            ops.ops.ROW_FUSE_ENABLED = True
    assert tuple(y_fused.shape) == (2, 64, 6, 4)
    assert (y_fused - y_eager).abs().max().item() <= 5e-5
    att = net.layers[0].att
    x = torch.randn(2, 24, 64).cuda()
    with torch.no_grad():
        xk, xv, _ = ops.q_shift_mix(x, [att.spatial_mix_k, att.spatial_mix_v, att.spatial_mix_r], 1, 0.25, (6, 4))
        k, v = att.key(xk), att.value(xv)
        y = ops.RUN_CUDA(att.spatial_decay / 24, att.spatial_first / 24, k, v)
    ref = clib.biwkv_fwd((att.spatial_decay / 24).detach().cpu().numpy(), (att.spatial_first / 24).detach().cpu().numpy(),
                         k.cpu().numpy(), v.cpu().numpy())
    assert np.abs(y.cpu().numpy() - ref).max() <= 1e-4 * np.sqrt((ref ** 2).mean())


@pytest.mark.gpu
def test_backbone_trains_through_the_hip_operators():
    import vision_rwkv_amd as ops
    torch.manual_seed(1)
    net = ops.VRWKV(img_size=32, embed_dims=64, depth=1).cuda()
    out = net(torch.randn(2, 3, 32, 32).cuda())
    out.square().mean().backward()
    g = net.layers[0].att.spatial_decay.grad
    assert g is not None and torch.isfinite(g).all() and g.abs().sum().item() > 0


def test_multihead_shift_tensor_ops_match_index_loops():
    """CPU: per-head Q-Shift by folding heads into the batch, against the index-loop oracle (with and without
    the trailing class token)."""
    import vision_rwkv_amd as ops
    from oracle import qshift
    rng = np.random.default_rng(3)
    for cls in (False, True):
        x = rng.standard_normal((2, 4 * 3 + int(cls), 128)).astype(np.float32)
        got = ops.q_shift_multihead(torch.from_numpy(x), 1, 64, (4, 3), with_cls_token=cls).numpy()
        assert np.array_equal(got, qshift.q_shift_multihead_loops(x, 1, 64, (4, 3), with_cls_token=cls))


@pytest.mark.gpu
@pytest.mark.parametrize("cls", [False, True])
def test_vrwkv6_backbone_fused_equals_eager_and_trains(cls):
    import vision_rwkv_amd as ops
    torch.manual_seed(2)
    net = ops.VRWKV6(img_size=64, embed_dims=128, num_heads=2, depth=2, post_norm=True, init_values=0.1,
                     with_cls_token=cls, output_cls_token=cls).cuda()
    img = torch.randn(2, 3, 96, 64).cuda()
    net.eval()
    with torch.no_grad():
        y_fused = net(img)
        import copy
        y16_fused = copy.deepcopy(net).bfloat16()(img.bfloat16())
        for m in net.modules():
            if hasattr(m, "fused_shift"):
                m.fused_shift = False
        ops.ops.ROW_FUSE_ENABLED = False               # every element-wise step as PyTorch ops
        try:
            y_eager = net(img)
        finally:
            ops.ops.ROW_FUSE_ENABLED = True
    fm = y_fused[0] if cls else y_fused
    fe = y_eager[0] if cls else y_eager
    assert tuple(fm.shape) == (2, 128, 6, 4)
    assert (fm - fe).abs().max().item() <= 5e-5
    if cls:
        assert tuple(y_fused[1].shape) == (2, 128) and (y_fused[1] - y_eager[1]).abs().max().item() <= 5e-5
    # the bf16 model (fused 16-bit kernels, GroupNorm + gate among them) stays within bf16 rounding of the fp32 one
    f16 = (y16_fused[0] if cls else y16_fused).float()
    assert (f16 - fe).abs().max().item() <= 0.1 * fe.abs().max().item()
    net.train()
    out = net(img)
    (out[0] if cls else out).square().mean().backward()
    for name in ("time_decay", "time_faaaa", "time_maa_w1"):
        g = getattr(net.layers[0].att, name).grad
        assert g is not None and torch.isfinite(g).all(), name
    assert net.layers[0].att.time_faaaa.grad.abs().sum().item() > 0


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["vrwkv", "vrwkv_key_norm", "vrwkv6", "vrwkv6_cls"])
def test_every_parameter_gradient_fused_equals_tensor_ops(kind):
    """One training step of a two-block backbone on 3 x 140 (141) tokens in fp32: the gradient of every parameter
    with the element-wise steps on the HIP kernels and their hand-written backward kernels against the same model
    with those steps as PyTorch tensor ops under autograd (the WKV operators are the HIP ones in both).  More than
    128 rows, so the channel sums of every backward kernel span several partial rows.
    Tolerance: 2e-4 of each gradient's largest entry (fast exp / rcp in the gates, fp32 sums in another order)."""
    import vision_rwkv_amd as ops
    torch.manual_seed(4)
    if kind.startswith("vrwkv6"):
        cls = kind.endswith("cls")
        net = ops.VRWKV6(img_size=64, embed_dims=128, num_heads=2, depth=2, post_norm=True, init_values=0.1,
                         with_cls_token=cls, output_cls_token=cls).cuda()
    else:
        cls = False
        net = ops.VRWKV(img_size=64, embed_dims=128, depth=2, post_norm=not kind.endswith("key_norm"), init_values=0.1,
                        key_norm=kind.endswith("key_norm")).cuda()
    for prm in net.parameters():                      # layer scales and biases away from their initial values
        if prm.dim() == 1:
            prm.data.add_(0.1 * torch.randn_like(prm))
    img = torch.randn(3, 3, 224, 160).cuda()
    net.train()

    def grads():
        net.zero_grad(set_to_none=True)
        out = net(img)
        out = out[0] if cls else out
        (out * torch.linspace(-1, 1, out.numel(), device=out.device).view_as(out)).sum().backward()
        return {n: p.grad.clone() for n, p in net.named_parameters() if p.grad is not None}, out.detach()

    g_fused, y_fused = grads()
    for m in net.modules():
        if hasattr(m, "fused_shift"):
            m.fused_shift = False
    ops.ops.ROW_FUSE_ENABLED = False
    try:
        g_eager, y_eager = grads()
    finally:
        ops.ops.ROW_FUSE_ENABLED = True
    assert (y_fused - y_eager).abs().max().item() <= 1e-4 * y_eager.abs().max().item()
    assert set(g_fused) == set(g_eager) and len(g_fused) > 20
    worst = ("", 0.0)
    for name, ge in g_eager.items():
        err = (g_fused[name] - ge).abs().max().item() / max(ge.abs().max().item(), 1e-12)
        if err > worst[1]:
            worst = (name, err)
        assert err <= 2e-4, (name, err)
    print(f"  {kind}: {len(g_eager)} parameter gradients, worst {worst[0]} {worst[1]:.1e}")


@pytest.mark.parametrize("kind", ["vrwkv", "vrwkv6"])
def test_reference_checkpoint_keys_load(kind):
    """CPU: a state dict with the reference's key names (vrwkv.py:351-358 keeps the patch embedding as
    `patch_embed.projection.*`; whole-model checkpoints prefix `backbone.` and carry a head) loads into the
    backbone, including a position table trained on another grid."""
    import vision_rwkv_amd as ops
    torch.manual_seed(0)
    if kind == "vrwkv":
        mk = lambda img: ops.VRWKV(img_size=img, patch_size=16, embed_dims=64, depth=2, init_values=1e-5,
                                   post_norm=True, key_norm=True)
        expect = {"layers.0.att.spatial_decay", "layers.0.att.spatial_first", "layers.0.att.spatial_mix_k",
                  "layers.0.att.spatial_mix_v", "layers.0.att.spatial_mix_r", "layers.1.ffn.spatial_mix_k",
                  "layers.0.gamma1", "layers.0.ln0.weight", "layers.1.att.key_norm.weight", "ln1.weight", "pos_embed"}
    else:
        mk = lambda img: ops.VRWKV6(img_size=img, patch_size=16, embed_dims=128, depth=2, num_heads=2)
        expect = {"layers.0.att.time_maa_x", "layers.0.att.time_maa_w1", "layers.0.att.time_decay",
                  "layers.0.att.time_decay_w2", "layers.0.att.time_faaaa", "layers.0.att.ln_x.weight",
                  "layers.0.att.gate.weight", "layers.1.ffn.spatial_mix_r", "ln1.weight", "pos_embed"}
    src = mk(48)                                   # "pre-trained" on a 3x3 grid
    for p in src.parameters():
        torch.nn.init.normal_(p)
    own = src.state_dict()
    assert expect <= set(own)
    ckpt = {"state_dict": {"backbone." + k.replace("patch_embed.", "patch_embed.projection."): v.clone()
                           for k, v in own.items()}}
    ckpt["state_dict"]["head.fc.weight"] = torch.zeros(10, 64)
    dst = mk(32)                                   # built for a 2x2 grid
    res = dst.load_reference_state_dict(ckpt)
    assert not res.missing_keys and not res.unexpected_keys
    assert dst.patch_resolution == (3, 3)
    for k, v in dst.state_dict().items():
        assert torch.equal(v, own[k]), k
    bad = {"backbone.layers.0.att.no_such_parameter": torch.zeros(1)}
    with pytest.raises(KeyError):
        mk(32).load_reference_state_dict(bad)


def test_pos_embed_resize_restates_the_interpolation():
    """CPU: resize_pos_embed against a direct F.interpolate of the grid part (embed.py:6-47), with and without
    extra tokens, and the identity when the grids agree."""
    from vision_rwkv_amd.backbone import resize_pos_embed
    import torch.nn.functional as F
    torch.manual_seed(1)
    pe = torch.randn(1, 1 + 12, 8)
    out = resize_pos_embed(pe, (3, 4), (6, 5), "bicubic", num_extra_tokens=1)
    grid = pe[:, 1:].reshape(1, 3, 4, 8).permute(0, 3, 1, 2)
    ref = F.interpolate(grid, size=(6, 5), mode="bicubic", align_corners=False).flatten(2).transpose(1, 2)
    assert out.shape == (1, 31, 8) and torch.equal(out[:, :1], pe[:, :1]) and torch.allclose(out[:, 1:], ref)
    assert resize_pos_embed(pe[:, 1:], (3, 4), (3, 4)) is not None and resize_pos_embed(pe[:, 1:], (3, 4), (3, 4)).shape == (1, 12, 8)
    with pytest.raises(RuntimeError):
        resize_pos_embed(pe, (3, 4), (6, 5))


@pytest.mark.gpu
@pytest.mark.parametrize("src,dst,C,dtype", [((14, 14), (24, 32), 768, torch.float32), ((12, 12), (24, 24), 1024, torch.bfloat16),
                                             ((14, 14), (7, 9), 192, torch.float16), ((1, 3), (5, 1), 257, torch.float32),
                                             ((40, 30), (3, 4), 33, torch.bfloat16), ((5, 4), (50, 84), 2, torch.float32)])
def test_pos_embed_resize_kernel_against_the_interpolation_in_float64(src, dst, C, dtype):
    """Result and gradient of the resampling kernel, with an extra token in front (whose slice makes odd row pitches and
    offsets), against F.interpolate in float64: 16 products of weights of at most 1 and fp32 sample points (their rounding,
    84 * 2^-24, shifts a weight by at most 1.5 times as much); the gradient adds up to 16 * (dst/src) products."""
    from vision_rwkv_amd.backbone import resize_pos_embed
    import torch.nn.functional as F
    torch.manual_seed(2)
    n = src[0] * src[1]
    pe = torch.randn(1, 1 + n, C).to(dtype)
    g = torch.randn(1, 1 + dst[0] * dst[1], C).to(dtype)
    ref_in = pe.double().requires_grad_()
    grid = ref_in[:, 1:].reshape(1, *src, C).permute(0, 3, 1, 2)
    ref = F.interpolate(grid, size=dst, mode="bicubic", align_corners=False).flatten(2).transpose(1, 2)
    ref = torch.cat((ref_in[:, :1], ref), 1)
    gref, = torch.autograd.grad(ref, ref_in, g.double())
    x = pe.cuda().requires_grad_()
    out = resize_pos_embed(x, src, dst, "bicubic", num_extra_tokens=1)
    gx, = torch.autograd.grad(out, x, g.cuda())
    assert out.dtype == dtype and gx.dtype == dtype
    eps = {torch.float32: 2e-5, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for a, r in ((out, ref), (gx, gref)):
        assert (a.double().cpu() - r.detach()).abs().max() <= eps * max(1.0, r.abs().max().item())


@pytest.mark.gpu
@pytest.mark.parametrize("N,dtype", [(1024, torch.bfloat16), (4096, torch.bfloat16), (768, torch.float32),
                                     (3072, torch.float32), (64, torch.float16), (8192, torch.bfloat16),
                                     (768, torch.bfloat16), (2048, torch.bfloat16), (1032, torch.bfloat16)])
def test_row_fuse_against_oracle(N, dtype):
    """The fused row epilogues against the float64 row-by-row oracle (oracle/blocks.py) on the same (rounded) inputs:
    every pre / LayerNorm / post combination the blocks use, rows that do not fill a workgroup.
    Tolerance: 2e-3 of the row scale for fp32 I/O (fast exp / rcp in the gate), one 16-bit rounding otherwise."""
    import vision_rwkv_amd as ops
    from oracle import blocks
    dev = "cuda:0"
    torch.manual_seed(N)
    rows = (3, 7)                                   # 21 rows: the last workgroup is partial
    a = torch.randn(*rows, N, device=dev).to(dtype)
    o = torch.randn(*rows, N, device=dev).to(dtype)
    w, b, g = (torch.randn(N, device=dev).to(dtype) for _ in range(3))
    combos = [(ops.ops.PRE_NONE, ops.ops.POST_SIGMOID_GATE, True), (ops.ops.PRE_NONE, ops.ops.POST_SIGMOID_GATE, False),
              (ops.ops.PRE_RELU_SQ, ops.ops.POST_NONE, True), (ops.ops.PRE_RELU_SQ, ops.ops.POST_NONE, False),
              (ops.ops.PRE_NONE, ops.ops.POST_RESIDUAL, True), (ops.ops.PRE_NONE, ops.ops.POST_RESIDUAL, False),
              (ops.ops.PRE_NONE, ops.ops.POST_NONE, True)]
    tol = 2e-3 if dtype == torch.float32 else 1e-2
    for pre, post, ln in combos:
        for gamma in ((g, None) if post == ops.ops.POST_RESIDUAL else (None,)):
            with torch.no_grad():
                got = ops.row_fuse(a, o if post else None, w if ln else None, b if ln else None, gamma, pre, post)
            f = lambda t: t.double().cpu().numpy() if t is not None else None
            ref = blocks.row_epilogue(f(a), f(o), f(w) if ln else None, f(b) if ln else None, f(gamma), pre, post)
            assert got.dtype == dtype and got.shape == a.shape
            err = np.abs(got.double().cpu().numpy() - ref).max() / max(np.abs(ref).max(), 1e-6)
            assert err <= tol, (pre, post, ln, gamma is not None, err)
            # the tensor-op sequence the blocks fall back to is the same function
            ft = lambda t: t.float() if t is not None else None
            seq = ops.row_fuse_tensor_ops(ft(a), ft(o), ft(w) if ln else None, ft(b) if ln else None, ft(gamma), pre, post)
            assert np.abs(seq.double().cpu().numpy() - ref).max() <= 2e-5 * max(np.abs(ref).max(), 1e-6)
    # a gradient is wanted: the tensor ops run and autograd works
    a2 = a.float().requires_grad_(True)
    ops.row_fuse(a2, o.float(), w.float(), b.float(), g.float(), ops.ops.PRE_NONE, ops.ops.POST_RESIDUAL).sum().backward()
    assert a2.grad is not None and torch.isfinite(a2.grad).all()


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,C,dtype", [(2, 5, 64, torch.bfloat16), (3, 197, 768, torch.bfloat16), (1, 7, 128, torch.float16),
                                          (2, 9, 192, torch.float32)])
def test_vrwkv6_mix_kernels_against_oracle(B, T, C, dtype):
    """maa_mix and groupnorm_gate against the float64 oracle (oracle/blocks.py) on the same (rounded) inputs.
    Tolerance: one 16-bit rounding of the result (1e-2 of the tensor's scale), 1e-5 for fp32 I/O."""
    import vision_rwkv_amd as ops
    from oracle import blocks
    dev = "cuda:0"
    f64 = lambda t: t.double().cpu().numpy()
    torch.manual_seed(C + T)
    x, sx = (torch.randn(B, T, C, device=dev).to(dtype) for _ in range(2))
    m = (0.3 * torch.randn(5, B, T, C, device=dev)).to(dtype)
    maas = [torch.rand(1, 1, C, device=dev).to(dtype) for _ in range(5)]
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    with torch.no_grad():
        got = ops.maa_mix(x, sx, m, maas)
    ref = blocks.maa_mix(f64(x), f64(sx), f64(m), [f64(a) for a in maas])
    seq = ops.ops.maa_mix_tensor_ops(x.float(), sx.float(), m.float(), [a.float() for a in maas])
    for g, r, sq in zip(got, ref, seq):
        assert g.dtype == dtype and np.abs(f64(g) - r).max() <= tol * np.abs(r).max()
        assert np.abs(f64(sq) - r).max() <= 1e-5 * np.abs(r).max()          # the tensor-op fallback is the same function
    if C % 64 == 0:
        H = C // 64
        for ydt in {torch.float32, dtype}:
            y = (3 * torch.randn(B, T, C, device=dev) + 1).to(ydt)
            gate = torch.randn(B, T, C, device=dev).to(dtype)
            w, b = torch.randn(C, device=dev).to(dtype), torch.randn(C, device=dev).to(dtype)
            with torch.no_grad():
                got = ops.groupnorm_gate(y, gate, w, b, H)
            ref = blocks.groupnorm_gate(f64(y), f64(gate), f64(w), f64(b), H)
            seq = ops.ops.groupnorm_gate_tensor_ops(y.float(), gate.float(), w.float(), b.float(), H)
            assert got.dtype == dtype and got.shape == gate.shape
            assert np.abs(f64(got) - ref).max() <= tol * np.abs(ref).max()
            assert np.abs(f64(seq) - ref).max() <= 1e-5 * np.abs(ref).max()
    # under autograd the tensor ops run
    xg = x.float().requires_grad_(True)
    sum(o.sum() for o in ops.maa_mix(xg, sx.float(), m.float(), [a.float() for a in maas])).backward()
    assert xg.grad is not None


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hp,Wp,C,head_dim,cls,dtype", [(2, 3, 5, 16, 0, False, torch.float32), (2, 14, 14, 192, 0, False, torch.float32),
                                                           (1, 7, 9, 22, 0, False, torch.float32), (2, 6, 4, 128, 64, True, torch.float32),
                                                           (2, 14, 14, 768, 0, False, torch.bfloat16), (3, 5, 3, 8, 0, False, torch.float32),
                                                           # many images: fewer, longer token chunks per workgroup (three
                                                           # chunks of 34 tokens; the whole image of 100 / 101 tokens)
                                                           (150, 10, 10, 256, 0, False, torch.bfloat16),
                                                           (300, 10, 10, 768, 0, False, torch.float32),
                                                           (240, 10, 10, 512, 64, True, torch.float16)])
def test_fused_qshift_mix_backward_against_autograd(B, Hp, Wp, C, head_dim, cls, dtype):
    """Gradients of the fused q_shift + mix (hand-written backward kernel) against autograd through the tensor-op
    formulation evaluated in float64 on the same inputs: grad of x and of every mix vector, three / two / one mix,
    per-head quarters with a trailing class token, a channel count that forces the scalar path, batches large enough
    for the kernel to take long token chunks.
    Tolerance: 1e-5 of the gradient's scale for fp32 I/O, 2e-2 for 16-bit I/O (one rounding of gx, 16-bit inputs)."""
    import vision_rwkv_amd as ops
    from vision_rwkv_amd.backbone6 import q_shift_multihead
    dev = "cuda:0"
    torch.manual_seed(Hp * Wp + C)
    T = Hp * Wp + (1 if cls else 0)
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    for n_mix in (3, 2, 1):
        x = torch.randn(B, T, C, device=dev).to(dtype).requires_grad_(True)
        mixes = [torch.rand(1, 1, C, device=dev).requires_grad_(True) for _ in range(n_mix)]
        gouts = [torch.randn(B, T, C, device=dev).to(dtype) for _ in range(n_mix)]
        outs = ops.q_shift_mix_autograd(x, mixes, 1, 0.25, (Hp, Wp), head_dim)
        torch.autograd.backward(outs, gouts)
        xr = x.detach().double().requires_grad_(True)
        mr = [m.detach().double().requires_grad_(True) for m in mixes]
        sx = (q_shift_multihead(xr, 1, head_dim, (Hp, Wp), cls) if head_dim else ops.q_shift(xr, 1, 0.25, (Hp, Wp)))
        ref = [xr * m + sx * (1 - m) for m in mr]
        torch.autograd.backward(ref, [g.double() for g in gouts])
        for o, r in zip(outs, ref):
            assert (o.double() - r).abs().max().item() <= tol * r.abs().max().item()
        assert (x.grad.double() - xr.grad).abs().max().item() <= tol * xr.grad.abs().max().item()
        for m, r in zip(mixes, mr):
            assert m.grad.shape == m.shape
            assert (m.grad.double() - r.grad).abs().max().item() <= tol * max(r.grad.abs().max().item(), 1.0)


@pytest.mark.gpu
@pytest.mark.parametrize("N,dtype,with_sums,rows", [
    (768, torch.float32, True, (5, 9)), (1024, torch.float32, True, (5, 9)), (64, torch.float32, True, (5, 9)),
    (768, torch.bfloat16, True, (5, 9)), (4096, torch.float32, False, (5, 9)), (3072, torch.bfloat16, False, (5, 9)),
    # more rows than the grid has waves (a wave walks several rows, the last ones fewer than the first), at every
    # vector shape the kernel picks: 8-byte x 3 (768 bf16), 16-byte x 2 (1024 bf16), 8-byte x 1 (192), 16-byte x 1 (384),
    # fp32 16-byte x 3 and x 4
    (768, torch.bfloat16, True, (3, 3001)), (1024, torch.bfloat16, True, (3, 2203)), (192, torch.bfloat16, True, (2, 4111)),
    (384, torch.float16, True, (2, 4111)), (768, torch.float32, True, (3, 2203)), (1024, torch.float32, True, (3, 1409)),
    # row lengths that leave the last group of lanes partly idle, one row, one vector per row
    (72, torch.bfloat16, True, (1, 1)), (200, torch.float16, True, (1, 513)), (1000, torch.bfloat16, True, (1, 33)),
    (520, torch.float32, True, (1, 7)), (4, torch.float32, True, (1, 4100))])
def test_row_fuse_backward_against_autograd(N, dtype, with_sums, rows):
    """Gradients of the fused row epilogues (hand-written backward kernel) against autograd through the tensor-op
    sequence in float64 on the same inputs: every pre / LayerNorm / post combination, on 45 rows (fewer than one row
    per wave) and on several thousand.  Rows longer than 1024 channels are differentiated by the kernel only
    without LayerNorm and gamma.  Tolerance: 2e-4 of each gradient's scale for fp32 I/O (fast exp / rcp in the gate,
    fp32 sums over rows), 3e-2 for 16-bit I/O."""
    import vision_rwkv_amd as ops
    O = ops.ops
    dev = "cuda:0"
    torch.manual_seed(N)
    tol = 2e-4 if dtype == torch.float32 else 3e-2
    combos = [(O.PRE_NONE, O.POST_SIGMOID_GATE, False, False), (O.PRE_RELU_SQ, O.POST_NONE, False, False),
              (O.PRE_NONE, O.POST_RESIDUAL, False, False)]
    if with_sums:
        combos += [(O.PRE_NONE, O.POST_SIGMOID_GATE, True, False), (O.PRE_RELU_SQ, O.POST_NONE, True, False),
                   (O.PRE_NONE, O.POST_RESIDUAL, True, True), (O.PRE_NONE, O.POST_RESIDUAL, False, True),
                   (O.PRE_NONE, O.POST_NONE, True, False), (O.PRE_RELU_SQ, O.POST_SIGMOID_GATE, True, False)]
    for pre, post, ln, use_gamma in combos:
        a = torch.randn(*rows, N, device=dev).to(dtype).requires_grad_(True)
        o = torch.randn(*rows, N, device=dev).to(dtype).requires_grad_(True) if post else None
        w = (1 + 0.3 * torch.randn(N, device=dev)).to(dtype).requires_grad_(True) if ln else None
        b = (0.3 * torch.randn(N, device=dev)).to(dtype).requires_grad_(True) if ln else None
        gm = torch.randn(N, device=dev).to(dtype).requires_grad_(True) if use_gamma else None
        gout = torch.randn(*rows, N, device=dev).to(dtype)
        out = ops.row_fuse(a, o, w, b, gm, pre, post)
        assert out.grad_fn is not None and "RowFuse" in type(out.grad_fn).__name__
        out.backward(gout)
        d = lambda t: t.detach().double().requires_grad_(True) if t is not None else None
        a2, o2, w2, b2, g2 = d(a), d(o), d(w), d(b), d(gm)
        ref = O.row_fuse_tensor_ops(a2, o2, w2, b2, g2, pre, post)
        ref.backward(gout.double())
        assert (out.double() - ref).abs().max().item() <= tol * ref.abs().max().item()
        for name, t, r in (("a", a, a2), ("other", o, o2), ("weight", w, w2), ("bias", b, b2), ("gamma", gm, g2)):
            if t is None:
                continue
            assert t.grad is not None, (name, pre, post, ln)
            err = (t.grad.double() - r.grad).abs().max().item() / max(r.grad.abs().max().item(), 1e-6)
            assert err <= tol, (name, pre, post, ln, use_gamma, err)


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,C,dtype", [(2, 5, 64, torch.float32), (3, 37, 768, torch.float32), (2, 23, 768, torch.bfloat16),
                                          (1, 7, 128, torch.float16),
                                          # hundreds and thousands of rows: many partial rows of the channel sums
                                          (1, 129, 256, torch.float32), (5, 300, 768, torch.float16), (64, 196, 768, torch.bfloat16),
                                          (3, 1000, 1024, torch.float32)])
def test_vrwkv6_mix_backward_against_autograd(B, T, C, dtype):
    """Gradients of maa_mix and groupnorm_gate (hand-written backward kernels) against autograd through the tensor-op
    sequences in float64 on the same inputs (group statistics written out with mean / var: the library's group-norm
    backward is wrong beyond 128 rows on this stack, see the next test); row counts that leave the last workgroup
    partial, and the VRWKV6-B layer shape.
    Tolerance: 1e-4 of each gradient's scale for fp32 I/O, 3e-2 for 16-bit."""
    import vision_rwkv_amd as ops
    O = ops.ops
    dev = "cuda:0"
    torch.manual_seed(C + T)
    tol = 1e-4 if dtype == torch.float32 else 3e-2
    d = lambda t: t.detach().double().requires_grad_(True)

    def check(name, got, ref):
        err = (got.double() - ref).abs().max().item() / max(ref.abs().max().item(), 1e-6)
        assert err <= tol, (name, err)

    x = torch.randn(B, T, C, device=dev).to(dtype).requires_grad_(True)
    sx = torch.randn(B, T, C, device=dev).to(dtype).requires_grad_(True)
    m = (0.3 * torch.randn(5, B, T, C, device=dev)).to(dtype).requires_grad_(True)
    maas = [torch.rand(1, 1, C, device=dev).to(dtype).requires_grad_(True) for _ in range(5)]
    gouts = [torch.randn(B, T, C, device=dev).to(dtype) for _ in range(5)]
    outs = ops.maa_mix(x, sx, m, maas)
    assert "MaaMix" in type(outs[0].grad_fn).__name__
    torch.autograd.backward(outs, gouts)
    x2, sx2, m2, maas2 = d(x), d(sx), d(m), [d(a) for a in maas]
    ref = O.maa_mix_tensor_ops(x2, sx2, m2, maas2)
    torch.autograd.backward(ref, [g.double() for g in gouts])
    for o, r in zip(outs, ref):
        check("out", o, r.detach())
    check("gx", x.grad, x2.grad); check("gsx", sx.grad, sx2.grad); check("gm", m.grad, m2.grad)
    for a, a2 in zip(maas, maas2):
        assert a.grad.shape == a.shape
        check("gmaa", a.grad, a2.grad)

    if C % 64 == 0:
        H = C // 64
        for ydt in {torch.float32, dtype}:
            y = (3 * torch.randn(B, T, C, device=dev) + 1).to(ydt).requires_grad_(True)
            gate = torch.randn(B, T, C, device=dev).to(dtype).requires_grad_(True)
            w = (1 + 0.3 * torch.randn(C, device=dev)).to(dtype).requires_grad_(True)
            b = (0.3 * torch.randn(C, device=dev)).to(dtype).requires_grad_(True)
            gout = torch.randn(B, T, C, device=dev).to(dtype)
            out = ops.groupnorm_gate(y, gate, w, b, H)
            assert "GroupNormGate" in type(out.grad_fn).__name__
            out.backward(gout)
            y2, g2, w2, b2 = d(y), d(gate), d(w), d(b)
            ref = O.groupnorm_gate_tensor_ops(y2, g2, w2, b2, H)
            ref.backward(gout.double())
            check("out", out, ref.detach())
            assert y.grad.dtype == ydt
            check("gy", y.grad, y2.grad); check("ggate", gate.grad, g2.grad)
            check("gw", w.grad, w2.grad); check("gb", b.grad, b2.grad)


@pytest.mark.gpu
def test_groupnorm_gate_parameter_gradients_do_not_depend_on_the_library_group_norm():
    """ln_x's weight and bias gradients over 200 rows: the kernel and the tensor-op path (which autograd differentiates
    when the kernel does not apply) against the sums written out in float64, g_w = sum_rows gout silu(gate) xh and
    g_b = sum_rows gout silu(gate).  torch.nn.functional.group_norm's own backward on this GPU stack returns other
    values beyond 128 rows (reported, not asserted: a fixed library would make that an error); neither path uses it."""
    import vision_rwkv_amd as ops
    O = ops.ops
    dev = "cuda:0"
    torch.manual_seed(11)
    rows, C, H = 200, 256, 4
    y0 = torch.randn(1, rows, C, device=dev)
    gate0 = torch.randn(1, rows, C, device=dev)
    w0, b0 = 1 + 0.3 * torch.randn(C, device=dev), 0.3 * torch.randn(C, device=dev)
    gout = torch.randn(1, rows, C, device=dev)
    yd = y0.double().reshape(rows, H, C // H)
    xh = ((yd - yd.mean(-1, keepdim=True)) / torch.sqrt(yd.var(-1, unbiased=False, keepdim=True) + 1e-5)).reshape(rows, C)
    gyn = gout.double().reshape(rows, C) * torch.nn.functional.silu(gate0.double().reshape(rows, C))
    want_w, want_b = (gyn * xh).sum(0), gyn.sum(0)
    rel = lambda a, r: ((a.double() - r).abs().max() / r.abs().max()).item()
    for name, fn in (("kernel", ops.groupnorm_gate), ("tensor ops", O.groupnorm_gate_tensor_ops)):
        y, gate, w, b = (t.clone().requires_grad_(True) for t in (y0, gate0, w0, b0))
        fn(y, gate, w, b, H, 1e-5).backward(gout)
        assert rel(w.grad, want_w) <= 1e-5 and rel(b.grad, want_b) <= 1e-5, (name, rel(w.grad, want_w), rel(b.grad, want_b))
    y, w, b = (t.clone().requires_grad_(True) for t in (y0, w0, b0))
    (torch.nn.functional.group_norm(y.reshape(rows, C), H, w, b, 1e-5) * torch.nn.functional.silu(gate0.reshape(rows, C))).backward(gout.reshape(rows, C))
    print(f"  library group_norm backward on {rows} rows: weight gradient off by {rel(w.grad, want_w):.1e}, bias by {rel(b.grad, want_b):.1e}")


@pytest.mark.gpu
def test_split_weight_gradient_of_the_block_projections():
    """The bias-free projections of a block under autograd with many tokens (backbone._proj, backbone._matmul): the
    weight gradient is a sum of batched partial products over the tokens; forward and input gradient are the plain
    GEMMs (bit-identical), the weight gradient agrees with the float32 product as well as the library's own bf16 GEMM
    does.  Few tokens, a bias or fp32 take the plain path."""
    from vision_rwkv_amd import backbone as bb
    dev = "cuda:0"
    torch.manual_seed(3)
    lin = torch.nn.Linear(192, 320, bias=False).to(dev).bfloat16()
    x = torch.randn(8, 1024, 192, device=dev).bfloat16().requires_grad_(True)
    g = torch.randn(8, 1024, 320, device=dev).bfloat16()
    y1 = bb._proj(lin, x)
    assert y1.grad_fn is not None and "SplitKLinear" in type(y1.grad_fn).__name__
    y1.backward(g)
    gx1, gw1 = x.grad.clone(), lin.weight.grad.clone()
    x.grad = None
    lin.weight.grad = None
    y2 = lin(x)
    y2.backward(g)
    assert torch.equal(y1, y2) and torch.equal(gx1, x.grad)
    ref = g.float().reshape(-1, 320).t() @ x.detach().float().reshape(-1, 192)
    scale = ref.abs().max()
    err_split = ((gw1.float() - ref).abs().max() / scale).item()
    err_plain = ((lin.weight.grad.float() - ref).abs().max() / scale).item()
    assert err_split <= max(2 * err_plain, 4e-3), (err_split, err_plain)
    w = (torch.randn(192, 40, device=dev) * 0.05).bfloat16().requires_grad_(True)
    z = bb._matmul(x.detach(), w)
    assert "SplitKMatmul" in type(z.grad_fn).__name__
    gz = torch.randn_like(z)
    z.backward(gz)
    refw = x.detach().float().reshape(-1, 192).t() @ gz.float().reshape(-1, 40)
    assert ((w.grad.float() - refw).abs().max() / refw.abs().max()).item() <= 4e-3
    # the stacked low-rank matrices of VRWKV6 (vrwkv6.py:184-185): x (5, B*T, 32) as the transposed view the block forms
    lo = (torch.randn(8 * 1024, 5, 32, device=dev) * 0.3).bfloat16().transpose(0, 1).requires_grad_(True)
    w2 = (torch.randn(5, 32, 192, device=dev) * 0.05).bfloat16().requires_grad_(True)
    m1 = bb._bmm(lo, w2)
    assert "SplitKBmm" in type(m1.grad_fn).__name__
    gm = torch.randn_like(m1)
    m1.backward(gm)
    glo1, gw21 = lo.grad.clone(), w2.grad.clone()
    lo.grad = None
    w2.grad = None
    m2 = torch.bmm(lo, w2)
    m2.backward(gm)
    assert torch.equal(m1, m2) and torch.equal(glo1, lo.grad)
    refw2 = torch.bmm(lo.detach().float().transpose(1, 2), gm.float())
    err_split = ((gw21.float() - refw2).abs().max() / refw2.abs().max()).item()
    err_plain = ((w2.grad.float() - refw2).abs().max() / refw2.abs().max()).item()
    assert err_split <= max(2 * err_plain, 4e-3), (err_split, err_plain)
    # the partial products are added by one sum over 16-bit values: it accumulates in fp32 and rounds once
    part = torch.randn(8, 320, 192, device=dev).bfloat16()
    assert torch.equal(part.sum(0), part.sum(0, dtype=torch.float32).to(torch.bfloat16))
    # plain paths
    small = torch.randn(2, 16, 192, device=dev).bfloat16().requires_grad_(True)
    assert "SplitK" not in type(bb._proj(lin, small).grad_fn).__name__
    assert "SplitK" not in type(bb._bmm(lo[:, :64], w2).grad_fn).__name__
    with torch.no_grad():
        assert bb._proj(lin, x).grad_fn is None


def _small_backbone(kind, C, dtype, key_norm, post_norm, cls, hw, device="cuda"):
    import vision_rwkv_amd as ops
    torch.manual_seed(11)
    kw = dict(img_size=hw[0] * 16, embed_dims=C, depth=2, key_norm=key_norm, post_norm=post_norm, init_values=0.3 if post_norm else None)
    net = ops.VRWKV6(num_heads=C // 64, with_cls_token=cls, **kw) if kind == "v6" else ops.VRWKV(**kw)
    with torch.no_grad():
        for n, p in net.named_parameters():
            if "time_maa_w" in n and p.dim() > 1 and n[-1] in "12" or "decay_w" in n:
                p.normal_(0, 0.02)
            elif p.dim() < 2 or p.shape[0] == 1:
                p.add_(0.05 * torch.randn_like(p))
    return net.to(device, dtype).eval()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [0, 1, 2, 4, 8, 16])
@pytest.mark.parametrize("kind,C,dtype,key_norm,post_norm,cls,hw,batch", [
    ("v4", 192, torch.bfloat16, False, False, False, (14, 14), 1), ("v4", 64, torch.float16, True, False, False, (1, 3), 24),
    ("v4", 416, torch.bfloat16, False, True, False, (7, 9), 3), ("v4", 256, torch.float16, True, True, False, (16, 15), 2),
    ("v6", 192, torch.bfloat16, False, False, True, (14, 14), 1), ("v6", 64, torch.float16, True, True, False, (1, 1), 96),
    ("v6", 384, torch.bfloat16, True, False, False, (9, 7), 3), ("v4", 160, torch.float32, True, False, False, (9, 7), 2),
    ("v4", 192, torch.float32, False, True, False, (14, 14), 1), ("v6", 192, torch.float32, True, False, True, (14, 13), 1),
    ("v6", 128, torch.float16, False, True, True, (5, 13), 2)])
def test_native_block_is_no_further_from_the_fp32_model_than_its_operators(kind, C, dtype, key_norm, post_norm, cls, hw, batch, tile):
    """Two blocks as native calls and operator by operator, both against the same weights and image in fp32.  The native call
    rounds at a subset of the places where the operators round, so its error may not exceed theirs.  Both norms are random:
    the errors of one token move together (one normalised vector: 1.4 apart for a single token of 64 channels), so a norm
    over n tokens scatters by about 1 / sqrt(2 n), their ratio by 1 / sqrt(n); with 65 or more tokens 1.25 is two of those
    at least."""
    net = _small_backbone(kind, C, dtype, key_norm, post_norm, cls, hw)
    img = torch.randn(batch, 3, hw[0] * 16, hw[1] * 16, device="cuda").to(dtype)
    from vision_rwkv_amd import ops as impl, option
    with torch.no_grad():
        x, res = net.embed(img)
        x = x if not cls else torch.cat((x, x[:, :1]), 1)
        assert all(l._native(x, res) is not None for l in net.layers)
        with option("linear_tile", tile):
            got = net(img).double()
        impl.BLOCK_FUSE_ENABLED = False
        try:
            assert net.layers[0]._native(x, res) is None
            plain = net(img).double()
            ref = net.float()(img.float()).double() if dtype != torch.float32 else plain
        finally:
            impl.BLOCK_FUSE_ENABLED = True
    if dtype == torch.float32:
        # two fp32 paths: products of up to 4 C = 768 terms, sqrt(768) 2^-24 = 1.7e-6 each, eight of them in a row and as
        # much again in VRWKV6's normalised, exponentiated decays
        assert (got - plain).norm() <= 2.8e-5 * plain.norm()
    else:
        assert (got - ref).norm() <= 1.25 * (plain - ref).norm()


@pytest.mark.gpu
@pytest.mark.parametrize("C,dtype,key_norm,post_norm,cls,hw,batch,segments", [
    (192, torch.bfloat16, False, False, False, (17, 18), 1, 0), (192, torch.float16, True, True, True, (24, 24), 1, 0),
    (64, torch.float32, True, False, True, (24, 24), 3, 0), (192, torch.float32, False, True, False, (17, 18), 1, 0),
    (768, torch.bfloat16, True, False, False, (28, 28), 2, 0), (128, torch.bfloat16, True, True, False, (5, 13), 3, 3),
    (64, torch.float16, False, False, True, (1, 33), 5, 2), (320, torch.float32, True, False, True, (8, 16), 2, 64)])
def test_native_v6_block_on_sequences_cut_into_segments(C, dtype, key_norm, post_norm, cls, hw, batch, segments):
    """Few long sequences, and short ones with a forced number of segments: the wkv6 operator inside the block exchanges states
    through its part of the block's workspace.  Held against the operators as above."""
    net = _small_backbone("v6", C, dtype, key_norm, post_norm, cls, hw)
    img = torch.randn(batch, 3, hw[0] * 16, hw[1] * 16, device="cuda").to(dtype)
    from vision_rwkv_amd import lib, ops as impl, option
    with torch.no_grad(), option("wkv6_segments", segments):
        assert lib().vrwkv_wkv6_fwd_workspace_bytes(batch, hw[0] * hw[1] + cls, C, C // 64) > 0
        x, res = net.embed(img)
        x = x if not cls else torch.cat((x, x[:, :1]), 1)
        assert all(l._native(x, res) is not None for l in net.layers)
        got = net(img).double()
        impl.BLOCK_FUSE_ENABLED = False
        try:
            plain = net(img).double()
            ref = net.float()(img.float()).double() if dtype != torch.float32 else plain
        finally:
            impl.BLOCK_FUSE_ENABLED = True
    if dtype == torch.float32:
        assert (got - plain).norm() <= 2.8e-5 * plain.norm()
    else:
        assert (got - ref).norm() <= 1.25 * (plain - ref).norm()


@pytest.mark.gpu
@pytest.mark.parametrize("C,dtype,key_norm,fp32_vectors", [(64, torch.bfloat16, False, False), (192, torch.float16, True, False),
                                                           (320, torch.bfloat16, True, True), (768, torch.float32, True, False),
                                                           (960, torch.bfloat16, False, True)])
def test_native_v6_block_reads_its_weights_as_the_modules_hold_them(C, dtype, key_norm, fp32_vectors, monkeypatch):
    """The low-rank matrices and vectors laid out inside the call against the same block given them laid out by tensor ops:
    bit-identical results.  1 - time_maa_x rounds to its own type in both."""
    from vision_rwkv_amd import backbone6
    from vision_rwkv_amd.ops import block_forward
    net = _small_backbone("v6", C, dtype, key_norm, True, False, (5, 7))
    if fp32_vectors:
        for l in net.layers:
            for m, names in ((l.att, ["time_maa_" + n for n in "xwkvrg"] + ["time_faaaa"]), (l.ffn, ["spatial_mix_r"])):
                for n in names:
                    getattr(m, n).data = getattr(m, n).data.float()
    calls = []

    def both(x, w, params, **num):
        flat = lambda n: params[n].detach().reshape(-1)
        laid_out = {n: params[n].detach().transpose(-1, -2).contiguous() for n in ("maa_w1", "maa_w2", "decay_w1", "decay_w2")}
        laid_out.update({n: params[n].detach().float() for n in ("att_kn_w", "att_kn_b") if n in params}, u=flat("u").float(),
                        att_mix=torch.stack([torch.zeros(C, device="cuda"), (1 - flat("maa_x")).float()]),
                        ffn_mix=torch.stack([flat("ffn_mix_k").float(), flat("ffn_mix_r").float()]),
                        maa=torch.stack([flat("maa_" + n).float() for n in "wkvrg"]))
        got, want = block_forward(x, w, params, **num), block_forward(x, {**w, **laid_out}, **num)
        calls.append(bool(torch.isfinite(want).all()) and torch.equal(got, want))
        return got

    monkeypatch.setattr(backbone6, "block_forward", both)
    with torch.no_grad():
        net(torch.randn(2, 3, 80, 112, device="cuda").to(dtype))
    assert calls == [True, True]


@pytest.mark.gpu
@pytest.mark.parametrize("key_norm,cls", [(False, True), (True, False)])
def test_native_v6_block_sees_writes_through_data(key_norm, cls):
    """A write to p.data leaves the parameter's version and address alone; the next inference must use it all the same:
    bit-identical to a model that is loaded with the new values."""
    import copy
    net = _small_backbone("v6", 128, torch.bfloat16, key_norm, True, cls, (6, 5))
    fresh = copy.deepcopy(net)
    img = torch.randn(2, 3, 96, 80, device="cuda").bfloat16()
    with torch.no_grad():
        before = net(img)
        for l in net.layers:
            for p in l.parameters():
                p.data.copy_(p.data * 1.25 + 0.01)
        got = net(img)
        fresh.load_state_dict(net.state_dict())
        want = fresh(img)
    assert not torch.equal(got, before) and torch.equal(got, want)


@pytest.mark.parametrize("v6,dtype,M,C,called,recorded", [
    (False, torch.bfloat16, 196, 192, True, True), (False, torch.bfloat16, 3136, 384, True, True), (False, torch.bfloat16, 12544, 512, True, True),
    (False, torch.bfloat16, 784, 768, True, True), (False, torch.float16, 1568, 768, True, False), (False, torch.bfloat16, 392, 1024, True, True),
    (False, torch.bfloat16, 784, 1024, True, False), (False, torch.bfloat16, 3136, 1024, True, False), (False, torch.bfloat16, 6272, 1024, False, False),
    (False, torch.bfloat16, 12544, 768, False, False), (True, torch.bfloat16, 6272, 768, True, True), (True, torch.bfloat16, 3136, 1024, True, True),
    (True, torch.float16, 6272, 1024, True, True), (True, torch.bfloat16, 12544, 1024, False, False),
    (False, torch.float32, 3136, 384, True, False), (False, torch.float32, 1960, 512, True, False),
    (False, torch.float32, 1568, 512, True, True), (False, torch.float32, 3136, 448, True, True), (False, torch.float32, 6272, 512, True, True),
    (True, torch.float32, 2352, 512, True, True), (False, torch.float32, 392, 768, True, True),
    (False, torch.float32, 784, 768, True, False), (False, torch.float32, 1568, 768, False, False), (False, torch.float32, 3136, 768, True, True),
    (False, torch.float32, 784, 1024, False, False), (False, torch.float32, 1568, 1024, True, True), (True, torch.float32, 784, 768, True, True),
    (True, torch.float32, 1568, 768, True, True), (True, torch.float32, 1568, 1024, True, True), (False, torch.bfloat16, 1 << 21, 64, False, False)])
def test_native_blocks_where_they_measured_faster(v6, dtype, M, C, called, recorded, monkeypatch):
    """The rule against the measured points: called eagerly, and recorded into a graph (the last one: 32-bit offsets)."""
    from vision_rwkv_amd.backbone import _native_size
    x = torch.empty(1, M, C, dtype=dtype, device="meta")
    for capturing, want in ((False, called), (True, recorded)):
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
        assert _native_size(x, 4 * C, v6) == want


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,shapes,splits", [(1, ((8, 8),), 0), (31, ((256, 256),), 0), (32, ((264, 248), (8, 520)), 0), (127, ((256, 512),), 0), (161, ((200, 72),), 2),
                                             (4096, ((768, 768),) * 3, 0), (4099, ((512, 256), (256, 1024), (768, 192)), 0), (1000, ((256, 256),) * 5, 7),
                                             (321, ((4096, 4352),), 0), (12544, ((768, 768), (3072, 768)), 0)])
def test_weight_gradients_in_one_launch(M, shapes, splits, dtype):
    """Token counts around the slices of 32 and the turns of four, partial tiles, ranges that do not divide, more tiles than compute units, rows at
    pitches of their own.  Against float64: the result's rounding (half a unit in the last of 8 or 11 bits: 2^-8, 2^-11 at most) and M fp32 additions,
    M 2^-24 of the sum of magnitudes at most."""
    from vision_rwkv_amd import option
    from vision_rwkv_amd.ops import weight_grad_group
    torch.manual_seed(M)
    gs = [torch.randn(M, o + 8, device="cuda").to(dtype)[:, :o] for o, _ in shapes]
    xs = [torch.randn(M, i, device="cuda").to(dtype) for _, i in shapes]
    with option("wgrad_splits", splits):
        outs = weight_grad_group(gs, xs)
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for g, x, out in zip(gs, xs, outs):
        ref = g.double().t() @ x.double()
        mag = g.double().abs().t() @ x.double().abs()
        assert ((out.double() - ref).abs() <= unit * ref.abs() * 1.01 + M * 2.0 ** -24 * mag + 2.0 ** -24).all()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,C,dtype,hw,shift,batch,cls", [
    ("v4", 192, torch.bfloat16, (14, 14), 1, 1, False), ("v4", 64, torch.float16, (1, 3), 1, 5, False), ("v4", 64, torch.bfloat16, (3, 1), 1, 2, False),
    ("v4", 1024, torch.bfloat16, (5, 7), 2, 2, False), ("v4", 512, torch.float32, (6, 9), 1, 3, False), ("v4", 256, torch.float32, (4, 4), 3, 1, False),
    ("v4", 96, torch.bfloat16, (7, 2), 5, 2, False), ("v6", 192, torch.bfloat16, (14, 13), 1, 1, True), ("v6", 64, torch.float16, (1, 1), 1, 7, True),
    ("v6", 576, torch.bfloat16, (4, 9), 2, 2, False)])
def test_norm_shift_and_mixes_in_one_launch(kind, C, dtype, hw, shift, batch, cls):
    """Images whose rows and columns are shorter than a workgroup's four tokens or than the shift, class tokens, rows of one and two
    pieces a lane: a block natively (one launch for norm, shift and mixes) is bit for bit the block with those as two launches,
    which more images in the batch get (the tail of a batch that is past the size of the rule)."""
    from vision_rwkv_amd import lib
    net = _small_backbone(kind, C, dtype, False, False, cls, hw)
    for l in net.layers:
        l.att.shift_pixel = l.ffn.shift_pixel = shift
    T = hw[0] * hw[1] + cls
    many = 700000 // (T * C) // batch * batch + batch
    x = torch.randn(many, T, C, device="cuda").to(dtype)
    with torch.no_grad():
        for b in (0, many - batch):
            few = x[b:b + batch].contiguous()
            assert all(l._native(few, hw) is not None for l in net.layers)
        from vision_rwkv_amd import option
        with option("linear_tile", 1):                       # the same products in either
            assert net.layers[1]._native(x, hw) is not None
            whole = net.layers[1](x, hw)
            part = torch.cat([net.layers[1](x[b:b + batch].contiguous(), hw) for b in (0, many - batch)])
    assert torch.equal(torch.cat((whole[:batch], whole[many - batch:])), part)


@pytest.mark.gpu
@pytest.mark.parametrize("C,dtype,hw,shift,batch,key_norm", [
    (192, torch.bfloat16, (14, 14), 1, 1, False), (192, torch.float16, (5, 7), 2, 3, True), (64, torch.bfloat16, (1, 1), 1, 1, False),
    (64, torch.float16, (3, 1), 1, 7, False), (64, torch.bfloat16, (2, 8), 3, 33, False), (256, torch.bfloat16, (3, 24), 1, 2, False),
    (320, torch.bfloat16, (4, 4), 1, 5, False), (384, torch.float16, (11, 17), 1, 1, True), (512, torch.bfloat16, (5, 3), 1, 1, False)])
def test_norm_shift_and_mixes_inside_the_projections(C, dtype, hw, shift, batch, key_norm):
    """Tiles of 16 tokens across images and past the last one, rows of half a wave and more, up to all 64 rows a workgroup holds: bit for bit the block that
    forms them in front of the projections, which a forced tile does (one order of the products in either).  That the block by itself has them inside is
    what the switch says, which makes anything else an error."""
    from vision_rwkv_amd import option
    net = _small_backbone("v4", C, dtype, key_norm, False, False, hw)
    for l in net.layers:
        l.att.shift_pixel = l.ffn.shift_pixel = shift
    x = torch.randn(batch, hw[0] * hw[1], C, device="cuda").to(dtype)
    with torch.no_grad():
        for l in net.layers:
            got = l._native(x, hw)
            with option("linear_tile", 1):
                want = l._native(x, hw)
            assert got is not None and torch.equal(got, want)
            with option("linear_mix", 1):
                assert torch.equal(l._native(x, hw), want)
            with option("linear_mix", 2):
                assert torch.equal(l._native(x, hw), want)


@pytest.mark.gpu
@pytest.mark.parametrize("C,dtype,hw,batch,inside", [
    (64, torch.bfloat16, (2, 24), 1, True), (64, torch.bfloat16, (2, 25), 1, False),            # 64 and 66 rows of a workgroup
    (256, torch.bfloat16, (17, 13), 4, True), (256, torch.bfloat16, (15, 12), 5, False),        # 884 and 900 tokens: 58.0 and 59.0 million by channels^2
    (384, torch.float16, (7, 29), 1, False), (384, torch.float16, (29, 7), 1, True), (384, torch.float16, (17, 12), 1, False),      # 74 rows; 203 and 204 tokens
    (576, torch.bfloat16, (1, 1), 1, False), (192, torch.float32, (2, 2), 1, False)])
def test_which_blocks_have_norm_shift_and_mixes_inside_the_projections(C, dtype, hw, batch, inside):
    """The rule's limits, on either side, by the switch that makes the other choice an error."""
    from vision_rwkv_amd import option
    l = _small_backbone("v4", C, dtype, False, False, False, hw).layers[0]
    x = torch.randn(batch, hw[0] * hw[1], C, device="cuda").to(dtype)
    with torch.no_grad(), option("linear_mix", 1):
        if inside:
            assert l._native(x, hw) is not None
        else:
            with pytest.raises(RuntimeError, match="not inside the projections"):
                l._native(x, hw)


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [((8, 8),), ((72, 136), (64, 64), (8, 200)), ((768, 768), (3072, 768), (768, 3072), (192, 40), (40, 192))])
def test_weights_transposed_in_one_launch(shapes):
    from vision_rwkv_amd.ops import transposed
    ws = [torch.randn(*s, device="cuda").bfloat16() for s in shapes]
    for w, t in zip(ws, transposed(ws)):
        assert torch.equal(t, w.t())


def _norm_errors(got, plain, exact):
    return [((a.double() - e).norm() / e.norm(), (b.double() - e).norm() / e.norm()) for a, b, e in zip(got, plain, exact)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,C,hidden", [(1, 6001, 192, 768), (2, 900, 768, 768), (3, 1500, 256, 512), (1, 4097, 384, 1152)])
def test_projections_in_one_launch_and_channel_mix_against_float64(B, T, C, hidden, dtype, monkeypatch):
    """Values and every gradient of grouped projections and of a channel mix whose element-wise steps are epilogues, against float64 of the
    same 16-bit weights and inputs: the grouped path rounds at a subset of the places where the operators round (the weight
    gradients are the same code), so it is no further off than they are; both errors are random, 1.1 is far outside their scatter over
    10^5 elements and more."""
    from vision_rwkv_amd import backbone as bb
    monkeypatch.setattr(bb, "CHANNEL_MIX_TILES", 0)
    torch.manual_seed(T)
    d = "cuda"
    ffn = bb.VRWKV_ChannelMix(C, 2, 0, hidden_rate=1).to(d)
    ffn.key, ffn.value = torch.nn.Linear(C, hidden, bias=False, device=d), torch.nn.Linear(hidden, C, bias=False, device=d)
    ffn.to(dtype)
    lins = [torch.nn.Linear(C, C, bias=False, device=d).to(dtype) for _ in range(3)]
    xs = [torch.randn(B, T, C, device=d).to(dtype).requires_grad_() for _ in range(3)]
    gs = [torch.randn(B, T, C, device=d).to(dtype) for _ in range(4)]
    params = [l.weight for l in (*lins, ffn.key, ffn.receptance, ffn.value)]

    def run():
        ys = bb._projs(lins, xs) + [bb._channel_mix(ffn, xs[0], xs[1])]
        assert type(ys[0].grad_fn).__name__ == type(ys[1].grad_fn).__name__
        return ys[0].grad_fn.name(), ys[3].grad_fn.name(), [y.detach() for y in ys] + list(torch.autograd.grad(ys, xs + params, gs))

    n0, n3, got = run()
    assert "_Projections" in n0 and "_ChannelMix" in n3
    with torch.no_grad():                                    # without autograd: the same launches
        for a, b in zip(bb._projs(lins, xs) + [bb._channel_mix(ffn, xs[0], xs[1])], got):
            assert torch.equal(a, b)
    monkeypatch.setattr(bb, "_own_weights", lambda *a: None)
    n0, n3, plain = run()
    assert "_Projections" not in n0 and "_ChannelMix" not in n3
    x6, p6 = [x.detach().double().requires_grad_() for x in xs], [p.detach().double().requires_grad_() for p in params]
    ys = [x @ w.t() for x, w in zip(x6, p6)]
    ys.append(torch.sigmoid(x6[1] @ p6[4].t()) * ((x6[0] @ p6[3].t()).relu().square() @ p6[5].t()))
    exact = [y.detach() for y in ys] + list(torch.autograd.grad(ys, x6 + p6, [g.double() for g in gs]))
    for i, (a, b) in enumerate(_norm_errors(got, plain, exact)):
        assert a <= 1.1 * b, (i, a, b)


@pytest.mark.gpu
def test_projections_with_hooks_frozen_parts_and_second_derivatives():
    from vision_rwkv_amd import backbone as bb
    torch.manual_seed(3)
    d, C = "cuda", 192
    lins = [torch.nn.Linear(C, C, bias=False, device=d).bfloat16() for _ in range(3)]
    xs = [torch.randn(1, 6000, C, device=d).bfloat16().requires_grad_(i != 1) for i in range(3)]
    lins[2].weight.requires_grad_(False)
    ys = bb._projs(lins, xs)
    assert "_Projections" in ys[0].grad_fn.name()
    sum(y.float().square().sum() for y in ys).backward()
    assert xs[0].grad is not None and xs[1].grad is None and lins[1].weight.grad is not None and lins[2].weight.grad is None
    for add in ("register_forward_hook", "register_full_backward_hook"):
        fired = []
        handle = getattr(lins[1], add)(lambda *a: fired.append(1))
        ys = bb._projs(lins, xs)
        assert "_Projections" not in ys[0].grad_fn.name()
        handle.remove()
    # a gradient that is itself differentiated goes through tensor ops: d/dx of |dy/dx g|^2 of a relu^2 product
    ffn = bb.VRWKV_ChannelMix(C, 2, 0).to(d).bfloat16()
    x, r = (torch.randn(1, 22000, C, device=d).bfloat16().requires_grad_() for _ in range(2))
    y = bb._channel_mix(ffn, x, r)
    assert "_ChannelMix" in y.grad_fn.name()
    g, = torch.autograd.grad(y, x, torch.ones_like(y), create_graph=True)
    gg, = torch.autograd.grad(g.float().square().sum(), x)
    X, R = x.detach().double().requires_grad_(), r.detach().double()
    wk, wr, wv = (l.weight.detach().double() for l in (ffn.key, ffn.receptance, ffn.value))
    G, = torch.autograd.grad((torch.sigmoid(R @ wr.t()) * ((X @ wk.t()).relu().square() @ wv.t())).sum(), X, create_graph=True)
    GG, = torch.autograd.grad(G.square().sum(), X)
    assert (gg.double() - GG).norm() <= 3e-2 * GG.norm()      # some eight bf16 roundings of 2^-9 = 2e-3, each of a differing sign pattern


@pytest.mark.parametrize("v6,dtype,M,C,called,recorded", [
    (False, torch.bfloat16, 12544, 768, True, True), (False, torch.bfloat16, 1568, 768, True, False), (False, torch.float16, 12544, 192, True, True),
    (True, torch.bfloat16, 1568, 768, True, True), (True, torch.float16, 25088, 576, True, True), (False, torch.bfloat16, 12544, 640, False, False),
    (False, torch.bfloat16, 12544, 1024, False, False), (False, torch.float32, 12544, 768, False, False),
    (False, torch.bfloat16, 1 << 18, 768, False, False)])
def test_native_blocks_of_wide_tiles_where_they_measured_faster(v6, dtype, M, C, called, recorded, monkeypatch):
    """The rule against the measured points: called eagerly, and recorded into a graph (the last one: 32-bit offsets)."""
    from vision_rwkv_amd.backbone import _native_wide
    x = torch.empty(1, M, C, dtype=dtype, device="meta")
    for capturing, want in ((False, called), (True, recorded)):
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
        assert _native_wide(x, 4 * C, v6) == want


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,Ns", [(1, 192, (16,)), (127, 128, (256, 272)), (160, 192, (768, 768, 768)), (1793, 192, (528, 64)), (225, 384, (784,)),
                                    (449, 256, (240, 16, 512, 256, 32)), (24000, 192, (512,)), (20000, 128, (1024,)), (321, 1152, (32, 768))])
def test_linear_group_of_wide_tiles(M, K, Ns, dtype):
    """Partial tiles of tokens and channels, one and several rounds of workgroups, both counts of stages, every epilogue.  Against float64 of the
    same 16-bit operands: the result's rounding (2^-8, 2^-11 relative at most) and fp32 additions, two orders below it; half as much again of
    the largest value's rounding bounds each."""
    import ctypes
    from vision_rwkv_amd import _lib, lib, option
    torch.manual_seed(M + K)
    d, n = "cuda", len(Ns)
    A = [torch.randn(M, K + 8 * i, device=d).to(dtype)[:, :K] if i else torch.randn(M, K, device=d).to(dtype) for i in range(n)]
    A = [a if a.stride(0) % 8 == 0 else a.contiguous() for a in A]
    W = [(torch.randn(N, K, device=d) * K ** -0.5).to(dtype) for N in Ns]
    for epi, extras in ((0, ()), (1, ("gate",)), (0, ("gate", "vec", "res")), (4, ("vec",))):
        extra = [{"gate": torch.randn(M, N, device=d).to(dtype), "vec": torch.randn(N, device=d).to(dtype), "res": torch.randn(M, N, device=d).to(dtype)}
                 for N in Ns]
        out = [torch.full((M + 1, N), 7.0, device=d, dtype=dtype) for N in Ns]
        ps = (_lib.Linear * n)(*[_lib.Linear(a=a.data_ptr(), w=w.data_ptr(), out=o.data_ptr(), N=N, K=K, lda=a.stride(0), epi=epi,
                                             **{k: e[k].data_ptr() for k in extras}) for a, w, o, N, e in zip(A, W, out, Ns, extra)])
        with option("linear_tile", 16):
            _lib.check(lib().vrwkv_linear_group(ps, n, M, 1 if dtype == torch.bfloat16 else 2, torch.cuda.current_stream().cuda_stream))
        for a, w, o, e in zip(A, W, out, extra):
            ref = a.double() @ w.double().t()
            if epi & 1:
                ref = ref.relu().square()
            if "gate" in extras:
                ref = ref * torch.sigmoid(e["gate"].double())
            if "vec" in extras:
                ref = ref + e["vec"].double() if epi & 4 else ref * e["vec"].double()
            if "res" in extras:
                ref = ref + e["res"].double()
            unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
            assert (o[:M].double() - ref).abs().max() <= 1.5 * unit * max(ref.abs().max().item(), 1.0)
            assert (o[M] == 7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,C,batch,hw,native", [("v4", 768, 8, (14, 14), False), ("v6", 1024, 8, (28, 28), True), ("v6", 192, 1, (14, 14), True)])
def test_inference_recorded_into_a_graph(kind, C, batch, hw, native):
    """A forward recorded after an eager one, where the two take different routes (and where they do not): the tables that the
    recording forms are not found by a later eager call, and every replay on new images equals the eager call of its route."""
    from vision_rwkv_amd import ops as impl
    net = _small_backbone(kind, C, torch.bfloat16, False, False, False, hw)
    image = lambda: torch.randn(batch, 3, hw[0] * 16, hw[1] * 16, device="cuda").bfloat16()

    def eager(x, fuse):
        impl.BLOCK_FUSE_ENABLED = fuse
        try:
            return net(x)
        finally:
            impl.BLOCK_FUSE_ENABLED = True

    with torch.no_grad():
        x = image()
        assert net.layers[0]._native(net.embed(x)[0], hw) is not None
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            net(x)
        torch.cuda.synchronize()
        kept = [dict(m._eval_cache) for l in net.layers for m in (l.att, l.ffn) if kind == "v4"]
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = net(x)
        # the recording found every table it needed, or (VRWKV6) needed none
        assert kept == [dict(m._eval_cache) for l in net.layers for m in (l.att, l.ffn) if kind == "v4"] and all(kept)
        first = eager(x, native)                          # before any replay
        assert bool(torch.isfinite(first).all())
        for i in range(3):
            if i:
                x.copy_(image())
            graph.replay()
            torch.cuda.synchronize()
            want = eager(x, native)
            assert torch.equal(y, want) and (i or torch.equal(first, want))


def _as_buffer(module, name):
    value = getattr(module, name).detach()
    delattr(module, name)
    module.register_buffer(name, value)


class _Twice(torch.nn.Module):
    def forward(self, x):
        return 2 * x


_CHANGES = {
    "pruned ffn key": lambda b, nn: nn.utils.prune.l1_unstructured(b.ffn.key, "weight", 0.3),
    "weight norm": lambda b, nn: nn.utils.weight_norm(b.ffn.key),
    "spectral norm": lambda b, nn: nn.utils.spectral_norm(b.ffn.key),
    "parametrised ffn key": lambda b, nn: nn.utils.parametrize.register_parametrization(b.ffn.key, "weight", _Twice()),
    "pruned layer scale": lambda b, nn: nn.utils.prune.l1_unstructured(b, "gamma1", 0.3),
    "parametrised layer scale": lambda b, nn: nn.utils.parametrize.register_parametrization(b, "gamma2", _Twice()),
    "pruned att key": lambda b, nn: nn.utils.prune.l1_unstructured(b.att.key, "weight", 0.3),
    "pruned mix": lambda b, nn: nn.utils.prune.l1_unstructured(b.ffn, "spatial_mix_k", 0.3),
    "pruned norm": lambda b, nn: nn.utils.prune.l1_unstructured(b.ln1, "bias", 0.3),
    "ffn key as a buffer": lambda b, nn: _as_buffer(b.ffn.key, "weight"),
    "output as a buffer": lambda b, nn: _as_buffer(b.att.output, "weight"),
    "mix as a buffer": lambda b, nn: _as_buffer(b.ffn, "spatial_mix_r"),
    "decay as a buffer": lambda b, nn: _as_buffer(b.att, "time_decay" if hasattr(b.att, "time_decay") else "spatial_decay"),
    "bonus as a buffer": lambda b, nn: _as_buffer(b.att, "time_faaaa" if hasattr(b.att, "time_faaaa") else "spatial_first"),
    "norm as a buffer": lambda b, nn: _as_buffer(b.ln2, "weight"),
    "layer scale as a buffer": lambda b, nn: _as_buffer(b, "gamma2"),
    "no ffn norm": lambda b, nn: setattr(b, "ln2", nn.Identity()),
}


@pytest.mark.parametrize("kind", ["v4", "v6"])
@pytest.mark.parametrize("change", list(_CHANGES))
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_blocks_whose_weights_are_held_otherwise_run_their_operators(device, change, kind, monkeypatch):
    """Pruned, normed, parametrised weights and parameters made buffers are not what the native call could read: it declines
    (on the CPU asked with its first check stood in for), and the model computes what its operators compute."""
    import torch.nn.utils.parametrize, torch.nn.utils.prune
    from vision_rwkv_amd import ops as impl, backbone, backbone6
    net = _small_backbone(kind, 64, torch.float32, False, True, False, (3, 4), device)
    if device == "cpu":
        for m in (backbone, backbone6):
            monkeypatch.setattr(m, "block_takes", lambda x: True)
            monkeypatch.setattr(m, "block_forward", lambda *a, **kw: "native")
    x = torch.randn(2, 12, 64, device=device)
    with torch.no_grad():
        assert all(l._native(x, (3, 4)) is not None for l in net.layers)
        for l in net.layers:
            _CHANGES[change](l, torch.nn)
        assert all(l._native(x, (3, 4)) is None for l in net.layers)
        if device == "cuda" and change != "no ffn norm":
            img = torch.randn(2, 3, 48, 64, device="cuda")
            got = net(img)
            monkeypatch.setattr(impl, "BLOCK_FUSE_ENABLED", False)
            assert torch.equal(got, net(img))


@pytest.mark.parametrize("kind", ["v4", "v6"])
@pytest.mark.parametrize("part,name", [("att", "spatial_mix_k"), ("ffn", "spatial_mix_r"), ("att", "spatial_decay"), ("att", "spatial_first"),
                                       ("att", "time_maa_x"), ("att", "time_maa_g"), ("att", "time_faaaa"), ("att", "time_decay"),
                                       ("att", "time_maa_w2")])
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_native_block_declines_vectors_of_another_size_or_device(device, part, name, kind, monkeypatch):
    """The operators refuse a vector that has not one element per channel, or lies elsewhere than x; the native call, which
    would read past its end, is not to be made (and is stood in for here)."""
    from vision_rwkv_amd import backbone, backbone6
    net = _small_backbone(kind, 64, torch.float32, False, True, False, (3, 4), device)
    for m in (backbone, backbone6):
        monkeypatch.setattr(m, "block_takes", lambda x: True)
        monkeypatch.setattr(m, "block_forward", lambda *a, **kw: "native")
    block, x = net.layers[1], torch.randn(2, 12, 64, device=device)
    module = getattr(block, part)
    if not hasattr(module, name):
        return
    old = getattr(module, name)
    with torch.no_grad():
        for new in [torch.zeros(n, device=device) for n in (1, 32, 128)] + ([old.cpu()] if device == "cuda" else []):
            setattr(module, name, torch.nn.Parameter(new))
            try:
                assert block._native(x, (3, 4)) is None, tuple(new.shape)
            except RuntimeError as e:                     # vectors that do not stack: the operators' own refusal
                assert "equal size" in str(e) or "same device" in str(e)
        setattr(module, name, old)
        assert block._native(x, (3, 4)) == "native"


@pytest.mark.parametrize("copied", [False, True])
def test_kept_tables_follow_a_module_that_is_cast_away_and_back(copied):
    """Casting a module gives its parameters new memory, possibly where the old lay, and leaves their versions alone: the kept
    value must be rebuilt, also in a copy whose original is gone."""
    import copy
    from vision_rwkv_amd.backbone import eval_cached
    torch.manual_seed(12)
    for n in [500] * 50 + [3, 1000, 70000]:              # (the same address again in a third of the first kind)
        m = torch.nn.Linear(n, 1, bias=False)
        take = lambda m: eval_cached(m, "table", (m.weight,), None, lambda: m.weight.detach().clone())
        assert torch.equal(take(m), m.weight) and take(m) is take(m)
        if copied:
            m = copy.deepcopy(m)
        m.half().float()
        assert torch.equal(take(m), m.weight), n
        with torch.no_grad():
            m.weight.add_(1)
        assert torch.equal(take(m), m.weight), n


@pytest.mark.gpu
def test_native_block_leaves_changed_modules_to_their_own_code():
    net = _small_backbone("v4", 192, torch.bfloat16, False, False, False, (14, 14))
    img = torch.randn(1, 3, 224, 224, device="cuda").bfloat16()
    blk = net.layers[0]
    with torch.no_grad():
        x, res = net.embed(img)
        base = net(img)
        calls = []
        h = blk.att.key.register_forward_hook(lambda *a: calls.append(1))
        assert blk._native(x, res) is None
        assert torch.allclose(net(img), base, rtol=0.1, atol=0.1) and calls
        h.remove()
        blk.ffn.key = torch.nn.Linear(192, 768, bias=True).cuda().bfloat16()
        assert blk._native(x, res) is None and net.layers[1]._native(x, res) is not None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert net.layers[1]._native(x, res) is None
        assert net.layers[1]._native(x.transpose(0, 1).transpose(0, 1).expand(2, -1, -1), res) is None      # not contiguous
        net.layers[1].att.output.weight.data = net.layers[1].att.output.weight.data.t()                     # transposed storage
        assert net.layers[1]._native(x, res) is None
        net.layers[1].float()
        assert net.layers[1]._native(x, res) is None
    assert net.layers[1]._native(x.detach().requires_grad_(), res) is None                                  # autograd on


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [0, 1, 3])
@pytest.mark.parametrize("n,M,O,I,dtype", [(1, 1, 8, 8, torch.bfloat16), (1, 31, 8, 136, torch.float16), (1, 33, 128, 120, torch.bfloat16),
                                           (2, 300, 136, 264, torch.float16), (5, 1000, 32, 768, torch.bfloat16),
                                           (1, 4096, 160, 384, torch.bfloat16), (1, 4099, 1024, 1024, torch.float16)])
def test_weight_gradient_kernel_against_float64(n, M, O, I, dtype, splits):
    """a^T b over the tokens at tile edges and remainders, with rows in their own tensors, inside wider ones, at odd addresses
    and transposed: one rounding of the result (8 / 11 significant bits: at most 2^-8 / 2^-11 of the value) and fp32 sums of M terms (2^-24 M of the
    magnitudes' sum)."""
    from vision_rwkv_amd import option
    from vision_rwkv_amd.ops import weight_grad
    torch.manual_seed(5)
    a, b = (torch.randn(n, M, c, device="cuda").to(dtype) for c in (O, I))
    wide = torch.full((M, n, O + 24), float("nan"), device="cuda", dtype=dtype)
    wide[..., 8:8 + O] = a.transpose(0, 1)
    odd = torch.empty(n * M * I + 1, device="cuda", dtype=dtype)[1:].view(n, M, I).copy_(b)
    ref = a.double().transpose(1, 2) @ b.double()
    mag = a.double().abs().transpose(1, 2) @ b.double().abs()
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = unit * 1.01 * ref.abs() + (M + 4) * 2.0 ** -24 * mag + 1e-7
    with option("wgrad_splits", splits):
        outs = [weight_grad(a, b), weight_grad(wide[..., 8:8 + O].transpose(0, 1), odd),
                weight_grad(a, b.transpose(1, 2).contiguous().transpose(1, 2))]
        if n == 1:
            outs.append(weight_grad(a[0], b[0])[None])
    for got in outs:
        assert got.dtype == dtype and got.shape == ref.shape and bool(((got.double() - ref).abs() <= bound).all())


@pytest.mark.gpu
def test_weight_gradient_of_many_tokens_in_more_ranges():
    """200000 tokens into 96 x 40: 260 ranges, against float64 with the bound of the test above."""
    from vision_rwkv_amd import lib
    from vision_rwkv_amd.ops import weight_grad
    torch.manual_seed(6)
    M, O, I = 200003, 96, 40
    assert lib().vrwkv_wgrad_workspace_bytes(1, M, O, I) > 200 * O * I * 4
    a, b = (torch.randn(M, c, device="cuda").bfloat16() for c in (O, I))
    got = weight_grad(a, b).double()
    ref, mag = a.double().t() @ b.double(), a.double().abs().t() @ b.double().abs()
    assert bool(((got - ref).abs() <= 2.0 ** -8 * 1.01 * ref.abs() + (M + 4) * 2.0 ** -24 * mag + 1e-7).all())


@pytest.mark.parametrize("M,O,I,own", [(4096, 1024, 1024, True), (9408, 4096, 256, True), (12544, 1024, 1024, False), (25088, 1024, 768, False),
                                       (12544, 768, 768, True), (100352, 768, 768, True), (301056, 768, 768, False), (301056, 64, 768, True),
                                       (301056, 96, 96, True), (12544, 3072, 768, False), (6272, 2048, 512, True)])
def test_weight_gradients_where_they_measured_faster(M, O, I, own, monkeypatch):
    """The rule against the measured points: the kernel is asked, or the library's partial products (on tensors without data)."""
    from vision_rwkv_amd import backbone as bb
    monkeypatch.setattr(bb, "weight_grad", lambda a, b: "own")
    monkeypatch.setattr(bb, "_transformed", lambda: False)
    a, b = (torch.empty(M, c, dtype=torch.bfloat16, device="meta") for c in (O, I))
    with torch.no_grad():
        assert (isinstance(bb._token_product(a, b, 8), str)) == own


@pytest.mark.gpu
def test_second_derivative_of_a_projection_goes_through_tensor_ops():
    from vision_rwkv_amd.backbone import _SplitKLinear
    torch.manual_seed(6)
    x = torch.randn(4096, 64, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    w = torch.randn(64, 64, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    y = _SplitKLinear.apply(x, w, 8)
    gw, = torch.autograd.grad(y.float().square().sum(), w, create_graph=True)
    ggx, = torch.autograd.grad(gw.float().sum(), x)
    assert ggx.shape == x.shape and bool(torch.isfinite(ggx).all()) and ggx.abs().max() > 0


@pytest.mark.parametrize("kind", ["linear", "matmul", "bmm"])
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_weight_gradients_of_a_batch_of_cotangents(kind, device, monkeypatch):
    """is_grads_batched runs the backward of a projection on batched tensors, which have no memory of their own: tensor ops,
    the same gradients as one cotangent at a time (eight partial sums, each below half the largest value, and two results
    rounded to bf16, 2^-9 each: below 2^-6 of the largest)."""
    from vision_rwkv_amd import backbone as bb
    if device == "cpu":                              # stands in for the kernel, which needs addresses
        def product(a, b):
            a.data_ptr(), b.data_ptr()
            return (a.float().transpose(-1, -2) @ b.float()).to(a.dtype)
        monkeypatch.setattr(bb, "weight_grad", product)
    torch.manual_seed(7)
    mk = lambda *s: torch.randn(*s, device=device, dtype=torch.bfloat16)
    shape = (2,) if kind == "bmm" else ()
    x, w, gs = mk(*shape, 256, 64), mk(*shape, 64, 64).requires_grad_(), mk(3, *shape, 256, 64)
    fn = {"linear": bb._SplitKLinear, "matmul": bb._SplitKMatmul, "bmm": bb._SplitKBmm}[kind]
    y = fn.apply(x, w, 8)
    batched, = torch.autograd.grad(y, w, gs, is_grads_batched=True, retain_graph=True)
    single = torch.stack([torch.autograd.grad(y, w, g, retain_graph=True)[0] for g in gs])
    assert (batched.float() - single.float()).abs().max() <= 2.0 ** -6 * single.float().abs().max()


@pytest.mark.parametrize("adjoint", [False, True])
def test_table_resize_of_a_batch_of_cotangents(adjoint, monkeypatch):
    """The derivative of either map on a batch of cotangents: tensor ops, equal to one at a time (fp32, taps of 4 x 4)."""
    from vision_rwkv_amd import ops
    def launch(t, src, dst, adj):                    # stands in for the kernel, which needs addresses
        t.data_ptr()
        return ops._table_resize_ops(t, src, dst, adj)
    monkeypatch.setattr(ops, "_table_resize_launch", launch)
    torch.manual_seed(8)
    src, dst = (5, 7), (8, 6)
    (n, m) = (48, 35) if adjoint else (35, 48)
    t = torch.randn(1, n, 4, requires_grad=True)
    y = ops._TableResize.apply(t, src, dst, adjoint)
    gs = torch.randn(3, 1, m, 4)
    batched, = torch.autograd.grad(y, t, gs, is_grads_batched=True, retain_graph=True)
    mapped = torch.vmap(lambda g: torch.autograd.grad(y, t, g, retain_graph=True)[0])(gs)
    assert torch.equal(mapped, batched)
    for b, g in zip(batched, gs):
        single, = torch.autograd.grad(y, t, g, retain_graph=True)
        assert torch.allclose(b, single, rtol=1e-5, atol=1e-5)
        # the pair are each other's adjoint
        assert abs(float((y.detach() * g).sum() - (t.detach() * single).sum())) < 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n_mix,through,C,head,cls,shift", [(1, 1, 64, 64, 0, 1), (2, 2, 128, 64, 1, 1), (3, 1, 192, 0, 0, 1), (2, 1, 20, 0, 0, 2), (3, 2, 768, 0, 0, 1)])
def test_shift_backward_adds_the_other_uses_gradients(dtype, n_mix, through, C, head, cls, shift):
    """x's gradients from its other uses, added in the shift's backward kernel: what the kernel without them gives for fp32 inputs of the same
    values, plus those, rounded once (half a unit of the type; 2^-21 of the terms for the fp32 sums)."""
    from vision_rwkv_amd.ops import q_shift_mix_autograd
    g = torch.Generator(device="cuda").manual_seed(3)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    B, res = 3, (5, 7)
    T = 35 + cls
    x = rand(B, T, C).to(dtype).requires_grad_()
    mixes = [rand(C).to(dtype).requires_grad_() for _ in range(n_mix)]
    outs = q_shift_mix_autograd(x, mixes, shift, 1 / 4, res, head, through)
    assert len(outs) == n_mix + through and all(torch.equal(o, x) for o in outs[n_mix:])
    gs = [rand(B, T, C).to(dtype) for _ in outs]
    got = torch.autograd.grad(outs, [x, *mixes], gs, retain_graph=True)
    xf, mf = x.detach().float().requires_grad_(), [m.detach().float().requires_grad_() for m in mixes]
    want = torch.autograd.grad(q_shift_mix_autograd(xf, mf, shift, 1 / 4, res, head), [xf, *mf], [t.float() for t in gs[:n_mix]])
    full = want[0].double() + sum(t.double() for t in gs[n_mix:])
    size = want[0].abs() + sum(t.float().abs() for t in gs[n_mix:])
    unit = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    assert ((got[0].double() - full).abs() <= unit * full.abs() + 2.0 ** -21 * size + (6e-8 if dtype is torch.float16 else 0)).all()
    assert all(torch.equal(a, b.to(dtype)) for a, b in zip(got[1:], want[1:]))
    # a use that has no gradient, and only such uses
    some = torch.autograd.grad(outs[:n_mix], x, gs[:n_mix], retain_graph=True)[0]
    assert torch.equal(some, want[0].to(dtype))
    assert torch.equal(torch.autograd.grad(outs[-1], x, gs[-1], retain_graph=True)[0], gs[-1])
    # one that is to be differentiated again keeps its graph
    s = rand(B, T, C).to(dtype).requires_grad_()
    first = torch.autograd.grad((outs[-1] * s).sum(), x, create_graph=True)[0]
    assert torch.equal(torch.autograd.grad(first.sum(), s)[0], torch.ones_like(s))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["v4", "v6"])
@pytest.mark.parametrize("post", [True, False])
def test_residual_gradients_added_in_the_shift_are_those_of_autograd(kind, post):
    """Blocks whose residual branches go through the token shift against the same blocks called with hooks, which take x itself (fp32:
    1e-5 of the norm, a sum's rounding over two blocks)."""
    net = _small_backbone(kind, 64, torch.float32, post, True, False, (3, 4), "cuda")
    img = torch.randn(2, 3, 48, 64, device="cuda")
    def grads():
        net.zero_grad(set_to_none=True)
        out = net(img)
        out = out[0] if isinstance(out, tuple) else out
        (out * torch.linspace(-1, 1, out.numel(), device="cuda").view_as(out)).sum().backward()
        return out.detach(), [p.grad for p in net.parameters() if p.grad is not None]
    out, got = grads()
    seen = []
    handles = [m.register_forward_hook(lambda *a: seen.append(1)) for l in net.layers for m in (l.att, l.ffn)]
    ref, want = grads()
    [h.remove() for h in handles]
    assert len(seen) == 2 * len(net.layers) and torch.equal(out, ref) and len(got) == len(want)
    assert all((a - b).norm() <= 1e-5 * b.norm() + 1e-12 for a, b in zip(got, want))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,C,skip", [(1, 1, 64, 0), (3, 11, 768, 0), (2, 17, 65, 0), (4, 196, 192, 1), (64, 196, 768, 0), (1, 33, 8, 0), (2, 4000, 1024, 0)])
def test_vector_added_to_every_token_and_its_gradient(dtype, B, T, C, skip):
    """The vector's gradient against float64: half a unit of the type (fp16: its subnormals too) and, for fp32 sums of at most 8 row lanes of a
    chunk and 1024 chunks in 32 slices, 2^-24 of the summed sizes for each of 256 additions one after the other at most."""
    from vision_rwkv_amd.ops import add_to_tokens
    g = torch.Generator(device="cuda").manual_seed(5)
    vec = torch.randn(1, 1, C, generator=g, device="cuda").to(dtype).requires_grad_()
    x = torch.randn(B, T, C, generator=g, device="cuda").to(dtype).requires_grad_()
    gy = torch.randn(B * T * C + skip, generator=g, device="cuda").to(dtype)[skip:].view(B, T, C)
    y = add_to_tokens(vec, x)
    assert torch.equal(y, vec + x) and "AddToTokens" in type(y.grad_fn).__name__
    gv, gx = torch.autograd.grad(y, [vec, x], gy, retain_graph=True)
    want, size = gy.double().sum((0, 1), keepdim=True), gy.double().abs().sum((0, 1), keepdim=True)
    unit = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    assert torch.equal(gx, gy) and gv.shape == vec.shape and gv.dtype == dtype
    assert ((gv.double() - want).abs() <= unit * want.abs() + 256 * 2.0 ** -24 * size + (6e-8 if dtype is torch.float16 else 0)).all()
    twice = torch.autograd.grad((y * y).sum(), vec, create_graph=True)[0]
    assert torch.equal(torch.autograd.grad(twice.sum(), vec)[0], torch.full_like(vec, 2 * B * T))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,C", [(1, 1, 64), (1, 16, 128), (2, 33, 192), (3, 197, 384), (1, 2000, 768), (64, 196, 768), (2, 70, 1024)])
def test_mixes_with_their_low_rank_products_inside(dtype, B, T, C, monkeypatch):
    """Against the same steps in float64 from the same 16-bit values: m rounded to the type first (as a product's result is), then one rounding
    per result.  A gradient sum's fp32 terms add 2^-21 of their sizes; where m falls on a rounding boundary, its two neighbours differ
    by a unit of the type."""
    from vision_rwkv_amd.ops import maa_lora_mix
    g = torch.Generator(device="cuda").manual_seed(9)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype).requires_grad_()
    x, sx, lo, w2, maas = rand(B, T, C), rand(B, T, C), rand(B * T, 160), rand(5, 32, C), [rand(1, 1, C) for _ in range(5)]
    product = lambda a, b: torch.bmm(a.transpose(1, 2).contiguous(), b)
    outs = maa_lora_mix(x, sx, lo, w2, maas, product)
    with torch.no_grad():
        assert all(torch.equal(a, b) for a, b in zip(outs, maa_lora_mix(x, sx, lo, w2, maas, product)))
    gs = [torch.randn(B, T, C, generator=g, device="cuda").to(dtype) for _ in range(5)]
    got = torch.autograd.grad(outs, [x, sx, *maas], gs, retain_graph=True)
    glo, gw2 = torch.autograd.grad(outs, [lo, w2], gs, retain_graph=True)
    unit = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    tiny = 6e-8 if dtype is torch.float16 else 0.0
    d = lambda t: t.detach().double()
    stack = lo.detach().view(B * T, 5, 32).transpose(0, 1)
    exact = torch.bmm(d(stack), d(w2)).view(5, B, T, C)
    m = exact.to(dtype).double()
    off = 2 * unit * exact.abs() + 2.0 ** -20 * torch.bmm(d(stack).abs(), d(w2).abs()).view(5, B, T, C) + tiny      # of m, at most
    f, xx = torch.stack([d(a) for a in maas]).view(5, 1, 1, C) + m, d(sx) - d(x)
    G = torch.stack([d(t) for t in gs])
    near = lambda a, want, slack: ((d(a) - want).abs() <= unit * (want.abs() + slack) + slack + 2.0 ** -21 + tiny).all()
    for i in range(5):
        assert near(outs[i], d(x) + xx * f[i], xx.abs() * off[i] + 2.0 ** -21 * (d(x).abs() + (xx * f[i]).abs()))
    assert near(got[0], (G * (1 - f)).sum(0), (G.abs() * off).sum(0) + 2.0 ** -21 * (G.abs() * (1 + f.abs())).sum(0))
    assert near(got[1], (G * f).sum(0), (G.abs() * off).sum(0) + 2.0 ** -21 * (G.abs() * f.abs()).sum(0))
    gm = (G * xx).view(5, B * T, C)
    for i in range(5):
        want, size = gm[i].sum(0), gm[i].abs().sum(0)
        assert ((d(got[2 + i]).view(-1) - want).abs() <= unit * want.abs() + 2.0 ** -16 * size + tiny).all()
    gm16 = gm.to(dtype)
    for a, want, size in ((glo, torch.bmm(gm, d(w2).transpose(1, 2)).transpose(0, 1).reshape(lo.shape), torch.bmm(gm.abs(), d(w2).abs().transpose(1, 2)).transpose(0, 1).reshape(lo.shape)),
                          (gw2, torch.bmm(d(stack).transpose(1, 2), gm), torch.bmm(d(stack).abs().transpose(1, 2), gm.abs()))):
        assert ((d(a) - want).abs() <= unit * want.abs() + (unit + 2.0 ** -16) * size + tiny).all()      # gm rounded once before the products
    # to be differentiated again: tensor ops, the same values within their roundings, and a graph
    again = torch.autograd.grad(outs, x, gs, create_graph=True)[0]
    assert again.requires_grad and ((d(again) - d(got[0])).norm() <= 8 * unit * d(got[0]).norm())
    assert maa_lora_mix(x.float(), sx.float(), lo.float(), w2.float(), [a.float() for a in maas], product) is None
    assert maa_lora_mix(x[..., :60], sx[..., :60], lo, w2[..., :60], [a[..., :60] for a in maas], product) is None
    with torch.autocast("cuda"):
        assert maa_lora_mix(x, sx, lo, w2, maas, product) is None


@pytest.mark.gpu
@pytest.mark.parametrize("post", [True, False])
def test_model_with_mixes_inside_is_the_model_without(post, monkeypatch):
    """VRWKV6 blocks with the products inside the mixes against products of their own: the forward bit for bit, the gradients within bf16's
    rounding of two blocks."""
    from vision_rwkv_amd import backbone6
    net = _small_backbone("v6", 128, torch.bfloat16, False, post, True, (5, 7), "cuda").train()
    img = torch.randn(3, 3, 80, 112, device="cuda").bfloat16()
    def run():
        net.zero_grad(set_to_none=True)
        out = net(img)
        out = out[0] if isinstance(out, tuple) else out
        (out.float() * torch.linspace(-1, 1, out.numel(), device="cuda").view_as(out)).sum().backward()
        return out.detach(), {n: p.grad.double() for n, p in net.named_parameters() if p.grad is not None}
    out, got = run()
    monkeypatch.setattr(backbone6, "maa_lora_mix", lambda *a: None)
    ref, want = run()
    assert torch.equal(out, ref) and got.keys() == want.keys()
    assert all((got[n] - want[n]).norm() <= 3e-2 * want[n].norm() + 1e-9 for n in got), {n: ((got[n] - want[n]).norm() / want[n].norm()).item() for n in got}


MISFITS = [("key", (192, 768)), ("receptance", (192, 384)), ("value", (384, 384)), ("value", (1536, 384)), ("receptance", (384, 192)), ("receptance", (384, 768)),
           ("value", (768, 192)), ("value", (768, 768))]


def test_weights_that_do_not_fit_their_inputs_are_not_the_grouped_launchs():
    """The rule of the grouped launch for a channel mix of 384 channels and 768 hidden ones, every tensor but the device's name as on a
    GPU: every weight has its input's width."""
    from types import SimpleNamespace
    from vision_rwkv_amd.ops import linear_takes
    x = SimpleNamespace(shape=(2, 4096, 384), numel=lambda: 2 * 4096 * 384, is_cuda=True, dtype=torch.bfloat16, device=torch.device("cpu"))
    weight = lambda i, o: torch.zeros(o, i, dtype=torch.bfloat16)
    fits = dict(key=weight(384, 768), receptance=weight(384, 384), value=weight(768, 384))
    assert linear_takes(x, [fits["receptance"]] * 3)
    for wrong in (weight(192, 384), weight(768, 384), torch.zeros(384, dtype=torch.bfloat16)):
        assert not linear_takes(x, [fits["receptance"], wrong])
    rule = lambda ws: linear_takes(x, list(ws.values()), (384, 384, ws["key"].shape[0]))
    assert rule(fits)
    for name, size in MISFITS[:4]:
        assert not rule({**fits, name: weight(*size)}), (name, size)


@pytest.mark.gpu
@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("name,size", MISFITS)
def test_channel_mixes_whose_weights_do_not_fit_raise_as_the_operators_do(name, size, grad):
    """Layers replaced by ones of another width: what nn.Linear and the gate's product raise.  (384 channels, 768 hidden, 8192 tokens.)"""
    from vision_rwkv_amd import backbone as bb, ops
    d = "cuda"
    ffn = bb.VRWKV_ChannelMix(384, 2, 0, hidden_rate=2).to(d).bfloat16()
    x = torch.randn(2, 4096, 384, device=d).bfloat16().requires_grad_(grad)
    setattr(ffn, name, torch.nn.Linear(*size, bias=False, device=d).bfloat16())
    with torch.set_grad_enabled(grad):
        with pytest.raises(RuntimeError):
            bb._channel_mix(ffn, x, x)
        if name == "value" and size[0] == 768:               # ... and both of one other width
            ffn.receptance = torch.nn.Linear(384, size[1], bias=False, device=d).bfloat16()
            assert bb._channel_mix(ffn, x, x).shape == (2, 4096, size[1])
        lins = [torch.nn.Linear(i, 384, bias=False, device=d).bfloat16() for i in (384, size[0] if size[0] != 384 else 192)]
        with pytest.raises(RuntimeError):
            bb._projs(lins, [x, x])
        a, w = x.detach().view(-1, 384), lins[1].weight.detach()
        with pytest.raises(RuntimeError, match="must be"):
            ops.linear_group([dict(a=a, w=w)])
        with pytest.raises(RuntimeError, match="must be"):
            ops.linear_group([dict(a=a, w=lins[0].weight.detach(), gate=a[:, :192].contiguous())])


def test_a_level_of_forward_mode_differentiation_is_a_transform():
    from vision_rwkv_amd.ops import _transformed
    assert not _transformed()
    with torch.autograd.forward_ad.dual_level():
        assert _transformed()
    assert not _transformed()


@pytest.mark.gpu
@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("kind", ["v4", "v6"])
def test_tangents_pass_through_frozen_blocks_up_to_the_operators_refusal(kind, grad):
    """Forward-mode tangents with frozen weights, at a size of the grouped launches (384 channels, 3 x 4096 tokens): the projections' and a channel
    mix's are those of tensor ops (bf16: some ten roundings of 2^-9 in the mix), the operators refuse as they do on their own."""
    import torch.autograd.forward_ad as fw
    from vision_rwkv_amd import backbone as bb
    net = _small_backbone(kind, 384, torch.bfloat16, False, False, False, (64, 64))
    net.requires_grad_(False)
    block, hw = net.layers[1], (64, 64)
    x, t = (torch.randn(3, 4096, 384, device="cuda").bfloat16() for _ in range(2))
    lins = (block.att.key, block.att.value, block.att.receptance)
    with torch.set_grad_enabled(grad), fw.dual_level():
        dual = fw.make_dual(x, t)
        for lin, y in zip(lins, bb._projs(lins, [dual] * 3)):
            assert torch.equal(fw.unpack_dual(y).tangent, torch.nn.functional.linear(t, lin.weight))
        got = fw.unpack_dual(block.ffn(dual, hw)).tangent
        with pytest.raises((RuntimeError, NotImplementedError)):
            block.att(dual, hw)
        with pytest.raises((RuntimeError, NotImplementedError)):
            block(dual, hw)
    ffn = type(block.ffn)(**({} if kind == "v4" else dict(n_head=6)), n_embd=384, n_layer=2, layer_id=1, hidden_rate=4).double()
    ffn.load_state_dict({n: p.double().cpu() for n, p in block.ffn.state_dict().items()})
    _, want = torch.func.jvp(lambda z: ffn(z, hw), (x.double().cpu(),), (t.double().cpu(),))
    assert (got.double().cpu() - want).norm() <= 3e-2 * want.norm()


def _other_strides(t):
    return t.transpose(0, -1).contiguous().transpose(0, -1)


def _other_place(t):
    return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,C,hw,batch", [("v4", 384, (64, 64), 3), ("v6", 384, (64, 64), 3), ("v4", 192, (14, 14), 2), ("v6", 192, (14, 14), 2)])
@pytest.mark.parametrize("unpack", [_other_strides, _other_place])
@pytest.mark.parametrize("key_norm", [False, True])
def test_saved_tensors_may_come_back_with_other_strides(kind, C, hw, batch, unpack, key_norm):
    """Hooks on saved tensors promise the values, not the strides or the place: the gradients are those without hooks (12288 tokens
    of 384 channels: the sizes of the grouped launches).  Not bit for bit: the library's products take other kernels for operands that lie otherwise, so
    their results move by a rounding to bf16, 2^-9 of the value on average, some ten of which follow one another in a block: 3e-2.
    (Tensors of one column come back as they were: torch's LayerNorm reads its own statistics as dense.)"""
    net = _small_backbone(kind, C, torch.bfloat16, key_norm, True, False, hw)
    x = torch.randn(batch, hw[0] * hw[1], C, device="cuda").bfloat16()
    g = torch.randn_like(x)

    def grads(hooks):
        xs = x.clone().requires_grad_()
        with hooks:
            y = net.layers[1](xs, hw)
        return torch.autograd.grad(y, [xs, *net.layers[1].parameters()], g)

    want = grads(contextlib.nullcontext())
    got = grads(torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach(), lambda t: unpack(t) if t.dim() and t.shape[-1] > 1 else t))
    assert all((a - b).norm() <= 3e-2 * b.norm() for a, b in zip(got, want))


def test_batched_products_take_dense_right_operands(monkeypatch):
    """The batched products of the low-rank maps' gradients are given no transposed views on the right, which the library's 16-bit ones are not to be
    trusted with on this target."""
    from types import SimpleNamespace
    from vision_rwkv_amd import backbone as bb, ops
    seen, bmm = [], torch.bmm
    monkeypatch.setattr(torch, "bmm", lambda a, b: seen.append(b.is_contiguous()) or bmm(a, b))
    x, w = torch.randn(5, 24, 32, requires_grad=True), torch.randn(5, 32, 64)
    torch.autograd.grad(bb._SplitKBmm.apply(x, w, 8).sum(), x)
    B, T, C = 2, 3, 64
    saved = torch.randn(B, T, C), torch.randn(B, T, C), torch.randn(B * T, 160), torch.randn(5, 32, C), torch.randn(5, C)
    ctx = SimpleNamespace(saved_tensors=saved, needs_input_grad=[True] * 5, token_product=lambda a, b: a.transpose(1, 2) @ b)
    gx, gsx, glo, gw2, gtable, _ = ops._MaaLoraMix.backward(ctx, *torch.randn(5, B, T, C))
    assert glo.shape == (B * T, 160) and len(seen) == 4 and all(seen)


def test_weights_too_wide_to_transpose_are_not_the_grouped_launchs():
    from types import SimpleNamespace
    from vision_rwkv_amd.ops import linear_takes
    x = SimpleNamespace(shape=(4096, 1024), numel=lambda: 4096 * 1024, is_cuda=True, dtype=torch.bfloat16, device=torch.device("cpu"))
    for n, takes in ((65536, True), (65536 + 128, False)):
        assert linear_takes(x, [torch.zeros(n, 1024, dtype=torch.bfloat16)]) is takes


@pytest.mark.gpu
@pytest.mark.parametrize("C", [8192, 8320])
def test_channel_mixes_wider_than_the_gates_backward_kernel(C, monkeypatch):
    """Rows of 8192 channels and more: the gradients of the tensor ops (bf16 products of up to C terms with fp32 sums, each result rounded: three roundings
    of 2^-9 follow one another, 1e-2)."""
    from vision_rwkv_amd import backbone as bb, ops
    torch.manual_seed(3)
    ffn = bb.VRWKV_ChannelMix(C, 2, 0, hidden_rate=1).cuda().bfloat16()
    with torch.no_grad():
        for p in (ffn.key.weight, ffn.value.weight, ffn.receptance.weight):
            p.normal_(0, C ** -0.5)
    xs = [torch.randn(520, C, device="cuda").bfloat16().requires_grad_() for _ in range(2)]
    over = [*xs, ffn.key.weight, ffn.receptance.weight, ffn.value.weight]
    g = torch.randn(520, C, device="cuda").bfloat16()
    got = torch.autograd.grad(bb._channel_mix(ffn, *xs), over, g)
    monkeypatch.setattr(ops, "ROW_FUSE_ENABLED", False)
    want = torch.autograd.grad(bb._channel_mix(ffn, *xs), over, g)
    assert all((a - b).norm() <= 1e-2 * b.norm() for a, b in zip(got, want))


def test_a_compiled_module_is_called_as_it_is():
    """module.compile() changes what a call runs: neither a projection nor a mix is then taken apart."""
    from vision_rwkv_amd import backbone as bb
    lin = torch.nn.Linear(8, 8, bias=False)
    assert bb._as_built(lin, torch.nn.Linear)
    lin.compile()
    assert not bb._as_built(lin, torch.nn.Linear)


class _Adapted(torch.nn.Linear):
    def forward(self, x):
        return 2 * super().forward(x)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["subclass", "sequential", "backward hook", "global hook"])
def test_projections_that_do_more_than_multiply_are_called(kind):
    """4096 tokens in training, where a plain projection's weight gradient is split: replaced layers and hooked ones run their own call."""
    from torch.nn.modules import module as hooks
    from vision_rwkv_amd import backbone as bb
    lin = (_Adapted if kind == "subclass" else torch.nn.Linear)(192, 192, bias=False).cuda().bfloat16()
    x = torch.randn(4096, 192, device="cuda").bfloat16().requires_grad_()
    called, handle = [], None
    if kind == "backward hook":
        handle = lin.register_full_backward_hook(lambda m, gi, go: called.append(m) or None)
    elif kind == "global hook":
        handle = hooks.register_module_forward_hook(lambda m, i, o: called.append(m) or None)
    fn = torch.nn.Sequential(lin) if kind == "sequential" else lin
    try:
        y = bb._proj(fn, x)
        y.sum().backward()
    finally:
        if handle is not None:
            handle.remove()
    assert torch.equal(y, lin(x)) and (handle is None or lin in called)
