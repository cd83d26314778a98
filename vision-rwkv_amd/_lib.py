"""ctypes binding of libvrwkv_hip.so (the C ABI declared in include/vrwkv_hip.h).

The library is loaded from this directory; it is never compiled at import time and there
is no fallback: a missing library is a hard error.
"""
import ctypes
import importlib.util
import os
import subprocess
import warnings

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libvrwkv_hip.so")

VRWKV_F32, VRWKV_BF16, VRWKV_F16 = 0, 1, 2
STATUS_NAMES = {0: "OK", 1: "INVALID_ARG", 2: "UNSUPPORTED_DTYPE", 3: "UNSUPPORTED_SHAPE",
                4: "LAUNCH_FAILED", 5: "WORKSPACE_TOO_SMALL"}

_lib = None
_host = None


class BlockArgs(ctypes.Structure):
    """vrwkv_block_args of include/vrwkv_hip.h."""
    POINTERS_A = ("x", "out", "workspace")
    POINTERS_B = ("ln1_w", "ln1_b", "ln2_w", "ln2_b", "gamma1", "gamma2", "att_mix", "ffn_mix", "w", "u", "key", "value",
                  "receptance", "output", "att_kn_w", "att_kn_b", "ffn_key", "ffn_receptance", "ffn_value", "ffn_kn_w", "ffn_kn_b",
                  "gate", "maa", "maa_w1", "maa_w2", "decay", "decay_w1", "decay_w2", "gn_w", "gn_b")
    INTS = ("B", "T", "C", "hidden", "heads", "Hp", "Wp", "shift_pixel", "quarter", "post_norm", "dtype")
    FLOATS = ("ln1_eps", "ln2_eps", "att_kn_eps", "ffn_kn_eps", "gn_eps")
    _fields_ = ([(n, ctypes.c_void_p) for n in POINTERS_A] + [("workspace_bytes", ctypes.c_size_t)]
                + [(n, ctypes.c_void_p) for n in POINTERS_B] + [(n, ctypes.c_int) for n in INTS] + [(n, ctypes.c_float) for n in FLOATS])


class Linear(ctypes.Structure):
    """vrwkv_linear of include/vrwkv_hip.h."""
    POINTERS = ("a", "w", "out", "gate", "vec", "res", "raw")
    _fields_ = [(n, ctypes.c_void_p) for n in POINTERS] + [(n, ctypes.c_int) for n in ("N", "K", "lda", "epi")]


class Block6Params(ctypes.Structure):
    """vrwkv_block6_params of include/vrwkv_hip.h."""
    POINTERS = ("maa_w1", "maa_w2", "decay_w1", "decay_w2", "maa_x", "maa_w", "maa_k", "maa_v", "maa_r", "maa_g", "ffn_mix_k", "ffn_mix_r",
                "u", "att_kn_w", "att_kn_b")
    _fields_ = [(n, ctypes.c_void_p) for n in POINTERS] + [("fp32_vectors", ctypes.c_int)]


class VrwkvError(RuntimeError):
    """Non-zero status from the C ABI (mirrors the RuntimeError TORCH_CHECK raises at
    classification/mmcls_custom/models/backbones/cuda_new/bi_wkv.cpp:6-8)."""

    def __init__(self, status, message):
        super().__init__(f"vrwkv status {status} ({STATUS_NAMES.get(status, '?')}): {message}")
        self.status = status


class _NoHost:
    """What host() answers without the compiled module: None and False, with which the classes of ops.py go on by themselves."""
    @staticmethod
    def wkv(*args):
        return None

    wkv6 = block_forward = wkv

    @staticmethod
    def weights_fit(*args):
        return False


def _load_host(path):
    """The module at path, or an ImportError that says why it cannot be this process's."""
    if not os.path.exists(path):
        raise ImportError(f"{path} is missing")
    spec = importlib.util.spec_from_file_location("_host", path)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    built, here = module.torch_version, torch.__version__.split("+")[0]
    if built != here:                                        # it passes torch's own objects: another build's layout may differ
        raise ImportError(f"{path} was built with torch {built}, this is {here}")
    return module


def host():
    """The compiled module of csrc/host: the operators' host side in C++.  It belongs to the torch that it was built with; where it is missing or
    another's, the operators run through the classes of ops.py, the same kernels at more host time a call, after one warning."""
    global _host
    if _host is None:
        lib()
        try:
            _host = _load_host(os.path.join(_HERE, "_host.so"))
        except ImportError as e:
            warnings.warn(f"{e}: operators are called through Python, which takes longer (make -C vision-rwkv_amd/csrc builds it)", RuntimeWarning)
            _host = _NoHost
    return _host


def build(force=True):
    """Compile libvrwkv_hip.so for gfx950 and _host.so with the Makefile in csrc/ (hipcc cross-compiles
    without a GPU)."""
    cmd = ["make", "-C", os.path.join(_HERE, "csrc"), "-j8"]
    if force:
        cmd.append("-B")
    subprocess.run(cmd, check=True)
    return LIB_PATH


def _declare(lib):
    c = ctypes
    vp, fp, i, sz = c.c_void_p, c.c_void_p, c.c_int, c.c_size_t
    lib.vrwkv_version.argtypes = []
    lib.vrwkv_version.restype = i
    lib.vrwkv_last_error.argtypes = []
    lib.vrwkv_last_error.restype = c.c_char_p
    lib.vrwkv_set_option.argtypes = [c.c_char_p, i]
    lib.vrwkv_set_option.restype = i
    lib.vrwkv_get_option.argtypes = [c.c_char_p, c.POINTER(c.c_int)]
    lib.vrwkv_get_option.restype = i
    lib.vrwkv_biwkv_fwd_workspace_bytes.argtypes = [i, i, i, i]
    lib.vrwkv_biwkv_fwd_workspace_bytes.restype = sz
    lib.vrwkv_biwkv_fwd.argtypes = [fp, fp, vp, vp, vp, i, i, i, i, vp, sz, vp]
    lib.vrwkv_biwkv_fwd.restype = i
    lib.vrwkv_biwkv_fwd_gate.argtypes = [fp, fp, vp, vp, vp, vp, i, i, i, i, vp, sz, vp]
    lib.vrwkv_biwkv_fwd_gate.restype = i
    lib.vrwkv_biwkv_fwd_static_max_workspace_bytes.argtypes = []
    lib.vrwkv_biwkv_fwd_static_max_workspace_bytes.restype = sz
    lib.vrwkv_biwkv_fwd_static.argtypes = [fp, fp, vp, vp, vp, i, i, i, i, vp]
    lib.vrwkv_biwkv_fwd_static.restype = i
    lib.vrwkv_biwkv_bwd_workspace_bytes.argtypes = [i, i, i, i]
    lib.vrwkv_biwkv_bwd_workspace_bytes.restype = sz
    lib.vrwkv_biwkv_bwd.argtypes = [fp, fp, vp, vp, vp, fp, fp, vp, vp, i, i, i, i, vp, sz, vp]
    lib.vrwkv_biwkv_bwd.restype = i
    lib.vrwkv_wkv6_fwd_workspace_bytes.argtypes = [i, i, i, i]
    lib.vrwkv_wkv6_fwd_workspace_bytes.restype = sz
    lib.vrwkv_wkv6_fwd.argtypes = [vp, vp, vp, vp, fp, vp, i, i, i, i, i, i, i, vp, sz, vp]
    lib.vrwkv_wkv6_fwd.restype = i
    lib.vrwkv_wkv6_fwd_whole.argtypes = [vp, vp, vp, vp, fp, vp, i, i, i, i, i, i, i, vp]
    lib.vrwkv_wkv6_fwd_whole.restype = i
    lib.vrwkv_wkv6_fwd_phases_bytes.argtypes = [i, i, i]
    lib.vrwkv_wkv6_fwd_phases_bytes.restype = sz
    lib.vrwkv_wkv6_fwd_phases.argtypes = [vp, vp, vp, vp, vp, vp, i, i, i, i, vp, sz, vp]
    lib.vrwkv_wkv6_fwd_phases.restype = i
    lib.vrwkv_wkv6_bwd_workspace_bytes.argtypes = [i, i, i, i]
    lib.vrwkv_wkv6_bwd_workspace_bytes.restype = sz
    lib.vrwkv_wkv6_bwd.argtypes = [vp, vp, vp, vp, fp, fp, fp, fp, fp, fp, fp, i, i, i, i, i, i, i, vp, sz, vp]
    lib.vrwkv_wkv6_bwd.restype = i
    lib.vrwkv_wkv6_bwd_like_workspace_bytes.argtypes = [i, i, i, i, i, i]
    lib.vrwkv_wkv6_bwd_like_workspace_bytes.restype = sz
    lib.vrwkv_wkv6_bwd_like.argtypes = lib.vrwkv_wkv6_bwd.argtypes
    lib.vrwkv_wkv6_bwd_like.restype = i
    lib.vrwkv_qshift_mix.argtypes = [vp, fp, c.POINTER(c.c_void_p), i, i, i, i, i, i, i, i, i, i, vp]
    lib.vrwkv_qshift_mix.restype = i
    lib.vrwkv_qshift_mix_bwd_workspace_bytes.argtypes = [i, i, i, i]
    lib.vrwkv_qshift_mix_bwd_workspace_bytes.restype = sz
    lib.vrwkv_qshift_mix_bwd.argtypes = [vp, fp, c.POINTER(c.c_void_p), i, vp, fp, i, i, i, i, i, i, i, i, i, vp, sz, vp]
    lib.vrwkv_qshift_mix_bwd.restype = i
    lib.vrwkv_maa_lora_mix.argtypes = [vp, vp, vp, vp, fp, c.POINTER(c.c_void_p), c.c_longlong, i, i, vp]
    lib.vrwkv_maa_lora_mix.restype = i
    lib.vrwkv_maa_lora_mix_bwd_workspace_bytes.argtypes = [c.c_longlong, i]
    lib.vrwkv_maa_lora_mix_bwd_workspace_bytes.restype = sz
    lib.vrwkv_maa_lora_mix_bwd.argtypes = [vp, vp, vp, vp, fp, c.POINTER(c.c_void_p), vp, vp, vp, fp, c.c_longlong, i, i, vp, sz, vp]
    lib.vrwkv_maa_lora_mix_bwd.restype = i
    lib.vrwkv_column_sums_workspace_bytes.argtypes = [c.c_longlong, i]
    lib.vrwkv_column_sums_workspace_bytes.restype = sz
    lib.vrwkv_column_sums.argtypes = [vp, vp, c.c_longlong, i, i, vp, sz, vp]
    lib.vrwkv_column_sums.restype = i
    lib.vrwkv_qshift_mix_bwd_add.argtypes = [vp, fp, c.POINTER(c.c_void_p), i, c.POINTER(c.c_void_p), i, vp, vp, i, i, i, i, i, i, i, i, i, i, vp, sz, vp]
    lib.vrwkv_qshift_mix_bwd_add.restype = i
    lib.vrwkv_rowfuse.argtypes = [vp, vp, vp, vp, vp, vp, c.c_longlong, i, i, i, c.c_float, i, vp]
    lib.vrwkv_rowfuse.restype = i
    lib.vrwkv_rowfuse_bwd_workspace_bytes.argtypes = [c.c_longlong, i]
    lib.vrwkv_rowfuse_bwd_workspace_bytes.restype = sz
    lib.vrwkv_rowfuse_bwd.argtypes = [vp, vp, vp, vp, vp, vp, vp, vp, fp, c.c_longlong, i, i, i, c.c_float, i, vp, sz, vp]
    lib.vrwkv_rowfuse_bwd.restype = i
    lib.vrwkv_maa_mix.argtypes = [vp, vp, vp, fp, c.POINTER(c.c_void_p), c.c_longlong, i, i, vp]
    lib.vrwkv_maa_mix.restype = i
    lib.vrwkv_groupnorm_gate.argtypes = [vp, vp, vp, vp, vp, c.c_longlong, i, i, c.c_float, i, i, vp]
    lib.vrwkv_groupnorm_gate.restype = i
    lib.vrwkv_maa_mix_bwd_workspace_bytes.argtypes = [c.c_longlong, i]
    lib.vrwkv_maa_mix_bwd_workspace_bytes.restype = sz
    lib.vrwkv_maa_mix_bwd.argtypes = [vp, vp, vp, fp, c.POINTER(c.c_void_p), vp, vp, vp, fp, c.c_longlong, i, i, vp, sz, vp]
    lib.vrwkv_maa_mix_bwd.restype = i
    lib.vrwkv_groupnorm_gate_bwd_workspace_bytes.argtypes = [c.c_longlong, i]
    lib.vrwkv_groupnorm_gate_bwd_workspace_bytes.restype = sz
    lib.vrwkv_groupnorm_gate_bwd.argtypes = [vp, vp, vp, vp, vp, vp, vp, fp, c.c_longlong, i, i, c.c_float, i, i, vp, sz, vp]
    lib.vrwkv_groupnorm_gate_bwd.restype = i
    lib.vrwkv_pos_resize.argtypes = [vp, vp, i, i, i, i, i, i, i, vp]
    lib.vrwkv_pos_resize.restype = i
    lib.vrwkv_block_fwd_workspace_bytes.argtypes = [i, i, i, i, i, i]
    lib.vrwkv_block_fwd_workspace_bytes.restype = sz
    lib.vrwkv_block_fwd.argtypes = [c.POINTER(BlockArgs), vp]
    lib.vrwkv_block_fwd.restype = i
    lib.vrwkv_block6_fwd.argtypes = [c.POINTER(BlockArgs), c.POINTER(Block6Params), vp]
    lib.vrwkv_block6_fwd.restype = i
    lib.vrwkv_linear_group.argtypes = [c.POINTER(Linear), i, i, i, vp]
    lib.vrwkv_linear_group.restype = i
    lib.vrwkv_transpose_group.argtypes = [c.POINTER(vp), c.POINTER(vp), c.POINTER(i), c.POINTER(i), i, vp]
    lib.vrwkv_transpose_group.restype = i
    ll = c.c_longlong
    lib.vrwkv_wgrad_workspace_bytes.argtypes = [i, i, i, i]
    lib.vrwkv_wgrad_workspace_bytes.restype = sz
    lib.vrwkv_wgrad.argtypes = [vp, vp, vp, i, i, i, i, i, i, ll, ll, i, vp, sz, vp]
    lib.vrwkv_wgrad.restype = i
    lib.vrwkv_biwkv_fwd_as.argtypes = [vp, vp, i, c.c_float, vp, vp, vp, i, i, i, i, vp, sz, vp]
    lib.vrwkv_biwkv_fwd_as.restype = i
    lib.vrwkv_biwkv_bwd_as.argtypes = [vp, vp, i, c.c_float, vp, vp, vp, vp, vp, vp, vp, i, i, i, i, vp, sz, vp]
    lib.vrwkv_biwkv_bwd_as.restype = i
    pi, pv = c.POINTER(i), c.POINTER(vp)
    lib.vrwkv_wgrad_group_workspace_bytes.argtypes = [pi, pi, i, i]
    lib.vrwkv_wgrad_group_workspace_bytes.restype = sz
    lib.vrwkv_wgrad_group.argtypes = [pv, pv, pv, pi, pi, pi, pi, i, i, i, vp, sz, vp]
    lib.vrwkv_wgrad_group.restype = i
    for name in ("rowfuse_bwd", "qshift_mix_bwd", "groupnorm_gate_bwd", "biwkv_bwd"):
        like = getattr(lib, f"vrwkv_{name}_like")
        like.argtypes, like.restype = getattr(lib, f"vrwkv_{name}").argtypes, i
    return lib


def lib():
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise ImportError(
                f"{LIB_PATH} is missing: build it first (python -c 'import __graft_entry__ as g; g.build()' "
                "or make -C vision-rwkv_amd/csrc); there is no non-HIP fallback")
        _lib = _declare(ctypes.CDLL(LIB_PATH))
    return _lib


def get_option(name):
    """Value of a tuning / testing switch of the library (include/vrwkv_hip.h lists the names)."""
    out = ctypes.c_int(0)
    check(lib().vrwkv_get_option(name.encode(), ctypes.byref(out)))
    return out.value


def set_option(name, value):
    check(lib().vrwkv_set_option(name.encode(), int(value)))


class option:
    """with option("wkv6_fwd_scalar", 1): ...  -- sets a switch for the block and restores it afterwards."""

    def __init__(self, name, value):
        self.name, self.value = name, value

    def __enter__(self):
        self.old = get_option(self.name)
        set_option(self.name, self.value)
        return self

    def __exit__(self, *exc):
        set_option(self.name, self.old)
        return False


def check(status):
    if status != 0:
        raise VrwkvError(status, lib().vrwkv_last_error().decode("utf-8", "replace"))
