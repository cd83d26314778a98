"""Performance cases: what users of this package have it compute, through its public entry points.

A case is a dict of plain values.  `listed()` names the fixed ones, `draw(rng)` gives another one of the same ranges,
`prepare` makes what a program has in hand before the call, `run` is one pass, `work` its unavoidable bytes and
operations, `tolerance` how far two correct implementations of the same precision may lie apart.

Kinds
  biwkv_fwd / biwkv_train    RUN_CUDA(w, u, k, v), without / with the gradients of all four inputs
  wkv6_fwd / wkv6_train      RUN_CUDA_RWKV6(B, T, C, H, r, k, v, w, u), the same two ways
  vrwkv_infer / vrwkv_train  the VRWKV backbone: feature map of a batch of images / one forward and backward, every
  vrwkv6_infer / vrwkv6_train    gradient packed for the all-reduce; the same for VRWKV6
"""
import torch

import vision_rwkv_amd as vr

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
_BYTES = {"fp32": 4, "bf16": 2, "fp16": 2}
_DEV = "cuda"

# widths and heads of the T / S / B models, and of L (VRWKV only)
_WIDTHS = ((192, 3), (384, 6), (768, 12))


def listed():
    return [
        # one image through one layer of VRWKV-T: the smallest call, all latency
        dict(name="biwkv_fwd_tiny_one_image", kind="biwkv_fwd", B=1, T=196, C=192, dtype="fp32"),
        # the operator at VRWKV-B's classification shape in the reference's own precision (evaluation without autocast)
        dict(name="biwkv_fwd_base", kind="biwkv_fwd", B=64, T=196, C=768, dtype="fp32"),
        # one layer's operator in bf16 training of VRWKV-B: forward and backward
        dict(name="biwkv_train_base_bf16", kind="biwkv_train", B=64, T=196, C=768, dtype="bf16"),
        # detection fine-tuning: two images of about 1333 x 800, fp32 as the detection configs train
        dict(name="biwkv_train_dense", kind="biwkv_train", B=2, T=4150, C=768, dtype="fp32"),
        # VRWKV6-B's operator at inference: every tensor in the model's bf16, the decay logits too
        dict(name="wkv6_fwd_base_bf16", kind="wkv6_fwd", B=64, T=196, C=768, H=12, dtype="bf16", w_dtype="bf16"),
        # ... and in training
        dict(name="wkv6_train_base_bf16", kind="wkv6_train", B=64, T=196, C=768, H=12, dtype="bf16", w_dtype="bf16"),
        # dense prediction with VRWKV6-B: few, long sequences
        dict(name="wkv6_fwd_dense_bf16", kind="wkv6_fwd", B=2, T=4150, C=768, H=12, dtype="bf16", w_dtype="bf16"),
        # VRWKV6-S fine-tuned at 384 x 384 with a class token (24 * 24 + 1 tokens), fp32 as the reference calls the kernel
        dict(name="wkv6_train_small_384", kind="wkv6_train", B=8, T=577, C=384, H=6, dtype="fp32", w_dtype="fp32"),
        # one photo through VRWKV-T: a latency-bound service call
        dict(name="vrwkv_tiny_infer_one_image", kind="vrwkv_infer", C=192, depth=12, batch=1, height=224, width=224,
             dtype="bf16", key_norm=False, post_norm=False),
        # VRWKV-L at 384 x 384 (key_norm, post-norm, layer scale; position table interpolated from the 192 x 192 grid)
        dict(name="vrwkv_large_infer_384", kind="vrwkv_infer", C=1024, depth=24, batch=16, height=384, width=384,
             dtype="bf16", key_norm=True, post_norm=True),
        # one data-parallel worker's step of VRWKV-B / VRWKV6-B pre-training at 224 x 224
        dict(name="vrwkv_base_train", kind="vrwkv_train", C=768, depth=12, batch=64, height=224, width=224,
             dtype="bf16", key_norm=False, post_norm=True),
        dict(name="vrwkv6_base_train", kind="vrwkv6_train", C=768, H=12, depth=12, batch=64, height=224, width=224,
             dtype="bf16", key_norm=False, post_norm=True, cls_token=False),
    ]


def _log_int(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["biwkv_fwd", "biwkv_train", "wkv6_fwd", "wkv6_train",
                       "vrwkv_infer", "vrwkv_train", "vrwkv6_infer", "vrwkv6_train"])
    if kind.startswith("biwkv"):
        # tokens of a 7 x 7 grid up to a padded 1333 x 800 image; widths of the models, or any other
        T = _log_int(rng, 49, 4200)
        C = rng.choice([192, 256, 384, 512, 768, 1024]) if rng.random() < 0.7 else rng.randint(65, 1023)
        B = _log_int(rng, 1, max(1, min(64, 64 * 196 * 768 // (T * C))))
        return dict(kind=kind, B=B, T=T, C=C, dtype=rng.choice(["fp32", "bf16", "fp16"]))
    if kind.startswith("wkv6"):
        T = _log_int(rng, 49, 4200)
        H = rng.choice([3, 6, 12]) if rng.random() < 0.7 else rng.randint(1, 16)
        B = _log_int(rng, 1, max(1, min(64, 64 * 196 * 12 // (T * H))))
        dtype = rng.choice(["fp32", "bf16", "fp16"])
        return dict(kind=kind, B=B, T=T, C=64 * H, H=H, dtype=dtype, w_dtype=rng.choice([dtype, "fp32"]))
    C, H = rng.choice(_WIDTHS)
    height, width = 16 * rng.randint(7, 32), 16 * rng.randint(7, 32)
    tokens = (height // 16) * (width // 16)
    train = kind.endswith("train")
    dtype = rng.choice(["bf16", "bf16", "fp32"] if train else ["bf16", "fp16", "fp32"])
    cap = 64 * 196 * 768 * 768 // (8 if dtype == "fp32" else 1)          # fp32 products run at a fraction of the rate
    batch = _log_int(rng, 1, max(1, min(64, cap // (tokens * C * C), 64 * 196 // tokens)))
    case = dict(kind=kind, C=C, depth=12, batch=batch, height=height, width=width, dtype=dtype,
                key_norm=rng.random() < 0.3, post_norm=rng.random() < 0.5)
    if kind.startswith("vrwkv6"):
        case.update(H=H, cls_token=rng.random() < 0.3)
    return case


# ---- inputs -----------------------------------------------------------------------------------------------------------

def _biwkv_inputs(case, gen):
    """k, v: outputs of the key and value projections; w, u: the layer's decay and bonus over their trained range,
    divided by the token count as the block does."""
    B, T, C = case["B"], case["T"], case["C"]
    dt = _DTYPES[case["dtype"]]
    pos = torch.arange(C, device=_DEV) / max(C - 1, 1)
    zigzag = ((torch.arange(C, device=_DEV) + 1) % 3 - 1) * 0.5
    w = (-5 + 8 * pos ** (0.7 + 1.3 * torch.rand((), generator=gen, device=_DEV)) + _randn(gen, C) * 0.3) / T
    u = (-1.2 + zigzag + _randn(gen, C) * 0.3) / T
    k, v = _randn(gen, B, T, C), _randn(gen, B, T, C)
    return [t.to(dt) for t in (w, u, k, v)]


def _wkv6_inputs(case, gen):
    """r, k, v: outputs of the projections; w: decay logits, each channel's base value (from -6 to -1 over the width, as
    the model sets it up) plus the data-dependent part; u: the bonus per channel, kept in fp32 by the model."""
    B, T, C, H = case["B"], case["T"], case["C"], case["H"]
    dt, wdt = _DTYPES[case["dtype"]], _DTYPES[case["w_dtype"]]
    r, k, v = (_randn(gen, B, T, C).to(dt) for _ in range(3))
    pos = torch.arange(C, device=_DEV) / (C - 1)
    w = (-6 + 5 * pos ** (0.7 + 1.3 * torch.rand((), generator=gen, device=_DEV)) + _randn(gen, B, T, C) * 0.3).to(wdt)
    u = ((1 - pos) * 0.5 + _randn(gen, C) * 0.1).reshape(H, C // H)
    return [r, k, v, w, u]


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device=_DEV)


def _backbone(case, gen):
    """The model with the weights of one in training: the initialisation's ranges for the projections, layer scale and
    low-rank maps grown to where they act, every vector moved off its start."""
    C, depth = case["C"], case["depth"]
    kw = dict(img_size=192 if depth == 24 else 224, embed_dims=C, depth=depth, key_norm=case["key_norm"],
              post_norm=case["post_norm"], init_values=1e-5 if case["post_norm"] else None)
    with torch.device(_DEV):
        if case["kind"].startswith("vrwkv6"):
            net = vr.VRWKV6(num_heads=case["H"], with_cls_token=case["cls_token"], **kw)
        else:
            net = vr.VRWKV(**kw)
    with torch.no_grad():
        for name, p in net.named_parameters():
            leaf = name.split(".")[-1]
            if leaf in ("gamma1", "gamma2"):
                p.copy_(0.3 + 0.05 * _randn(gen, *p.shape))
            elif leaf in ("time_maa_w1", "time_maa_w2", "time_decay_w1", "time_decay_w2"):
                p.copy_(0.02 * _randn(gen, *p.shape))
            elif p.dim() >= 2 and leaf == "weight":
                p.copy_(_randn(gen, *p.shape) * p[0].numel() ** -0.5)
            elif leaf == "bias":
                p.copy_(0.02 * _randn(gen, *p.shape))
            else:
                p.add_(0.02 * _randn(gen, *p.shape))
    return net.to(_DTYPES[case["dtype"]])


def prepare(case, seed):
    gen = torch.Generator(device=_DEV).manual_seed(seed)
    kind = case["kind"]
    state = {"kind": kind}
    if kind.startswith(("biwkv", "wkv6")):
        inputs = (_biwkv_inputs if kind.startswith("biwkv") else _wkv6_inputs)(case, gen)
        if kind.endswith("train"):
            inputs = [t.requires_grad_() for t in inputs]
            # Bi-WKV returns its input's type, wkv6 fp32: the gradient that comes back is of that type
            state["gy"] = _randn(gen, case["B"], case["T"], case["C"])
            if kind.startswith("biwkv"):
                state["gy"] = state["gy"].to(_DTYPES[case["dtype"]])
        state["inputs"] = inputs
        state["shape"] = (case["B"], case["T"], case["C"], case.get("H"))
        return state
    net = _backbone(case, gen)
    dt = _DTYPES[case["dtype"]]
    state["images"] = _randn(gen, case["batch"], 3, case["height"], case["width"]).to(dt)
    if kind.endswith("train"):
        net.train()
        # what a dense head sends back: one gradient per feature
        state["gout"] = _randn(gen, case["batch"], case["C"], case["height"] // 16, case["width"] // 16).to(dt)
    else:
        net.eval()
    state["net"] = net
    state["buckets"] = _buckets(net)
    return state


def _buckets(net):
    """The parameters by their role, one list over the layers each: what a data-parallel worker packs together."""
    roles = {}
    for name, p in net.named_parameters():
        roles.setdefault(".".join(s for s in name.split(".") if not s.isdigit()), []).append(p)
    return list(roles.values())


# ---- one pass ---------------------------------------------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind.startswith(("vrwkv_", "vrwkv6_")):
        net = state["net"]
        if kind.endswith("infer"):
            with torch.no_grad():
                return net(state["images"])
        net.zero_grad(set_to_none=True)
        out = net(state["images"])
        out.backward(state["gout"])
        # the gradients leave as a worker hands them to its all-reduce: one flat bucket per role
        return [out.detach()] + [torch.cat([p.grad.flatten() for p in bucket]) for bucket in state["buckets"]]
    x = state["inputs"]
    if kind.startswith("biwkv"):
        def op():
            return vr.RUN_CUDA(*x)
    else:
        def op():
            return vr.RUN_CUDA_RWKV6(*state["shape"], *x)
    if kind.endswith("fwd"):
        with torch.no_grad():
            return op()
    y = op()
    return [y.detach()] + list(torch.autograd.grad(y, x, state["gy"]))


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------

def work(case):
    kind, es = case["kind"], _BYTES[case["dtype"]]
    if kind.startswith(("biwkv", "wkv6")):
        B, T, C = case["B"], case["T"], case["C"]
        n = B * T * C
        if kind.startswith("biwkv"):
            if kind.endswith("fwd"):
                return dict(bytes=3 * n * es + 2 * C * es, flops=29 * n)
            # k, v, gy read, y, gk, gv written; the backward's two scans are about twice the forward's
            return dict(bytes=6 * n * es + 4 * C * es, flops=3 * 29 * n)
        ws = _BYTES[case["w_dtype"]]
        scan = B * T * case["H"] * (10 * 64 * 64 + 3 * 64)
        if kind.endswith("fwd"):
            return dict(bytes=n * (3 * es + ws + 4) + 4 * C, flops=scan)
        # r, k, v, w, gy read; y, gr, gk, gv, gw written in their inputs' types
        return dict(bytes=n * (6 * es + 2 * ws + 8) + 8 * C, flops=3 * scan)
    C, depth = case["C"], case["depth"]
    tokens = case["batch"] * ((case["height"] // 16) * (case["width"] // 16) + (1 if case.get("cls_token") else 0))
    per_block = 14 * C * C + 448 * C if kind.startswith("vrwkv6") else 13 * C * C
    weights = depth * per_block + 768 * C
    features = tokens * C
    images = case["batch"] * 3 * case["height"] * case["width"]
    if kind.endswith("infer"):
        return dict(bytes=es * (weights + images + features), flops=2 * tokens * weights)
    return dict(bytes=es * (2 * weights + images + 2 * features), flops=6 * tokens * weights)


def tolerance(case):
    """About four times what was measured: the operators against the same formulas in float64, the backbones against the
    same model with every element-wise step left to tensor ops, at the same precision (and against the model in fp32)."""
    kind, dtype = case["kind"], case["dtype"]
    if kind.startswith(("biwkv", "wkv6")):
        # 16-bit results carry their own rounding (1.7e-3 / 2.1e-4 in the 2-norm, half a unit at most)
        if dtype != "fp32" and kind != "wkv6_fwd":
            return {"rel": 7e-3, "max": 1.6e-2} if dtype == "bf16" else {"rel": 8.5e-4, "max": 2.3e-3}
        if kind.startswith("biwkv"):
            return {"rel": 5e-6, "max": 5e-5}         # 1.2e-6 and 1.3e-5 measured
        if kind == "wkv6_fwd":
            return {"rel": 2e-5, "max": 2e-4}         # fp32 results whatever the inputs: 5.1e-6, 5.1e-5
        # the decay logits' gradient is a running difference of two nearly equal sums: 8.2e-5 and 9e-4 at 4200 tokens
        return {"rel": 3.3e-4, "max": 4e-3}
    v6, train = kind.startswith("vrwkv6"), kind.endswith("train")
    if dtype == "fp32":
        if v6:
            return {"rel": 7e-4, "max": 2e-2} if train else {"rel": 1e-4, "max": 1e-3}
        return {"rel": 1.2e-5, "max": 1.2e-4} if train else {"rel": 5e-6, "max": 3e-5}
    if dtype == "fp16":
        return {"rel": 1.2e-2}
    # bf16: 12 or 24 blocks of rounded activations; the worst gradient bucket
    if train:
        return {"rel": 0.18 if v6 else 0.09}          # 5.0e-2 (a token-mix bucket), 2.4e-2
    return {"rel": 6e-2}                              # 1.8e-2
