"""Host-side checks that need no GPU: the C-ABI library loads, exports every symbol the header
declares, and rejects bad arguments with a status and a message before touching the device."""
import ctypes
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    import vision_rwkv_amd
    if not os.path.exists(vision_rwkv_amd.LIB_PATH):
        vision_rwkv_amd.build(force=False)
    return vision_rwkv_amd.lib()


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "vrwkv_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(vrwkv_[a-z0-9_]+)\s*\(", text)))


def test_every_declared_symbol_is_exported(lib):
    names = declared_symbols()
    assert "vrwkv_biwkv_fwd" in names and "vrwkv_last_error" in names
    for n in names:
        assert hasattr(lib, n), f"{n} is declared in include/vrwkv_hip.h but not exported"


def test_version_and_error_string(lib):
    assert lib.vrwkv_version() >= 100
    assert isinstance(lib.vrwkv_last_error(), bytes)


def test_option_values_are_validated(lib):
    """vrwkv_set_option refuses unknown names and values the plans would silently ignore; accepted values read back."""
    val = ctypes.c_int(-1)
    assert lib.vrwkv_set_option(b"no_such_switch", 1) == 1
    assert lib.vrwkv_get_option(b"no_such_switch", ctypes.byref(val)) == 1
    for name, good, bad in ((b"biwkv_l", (4, 8, 16, 25, 28, 0), (7, 32, -1)), (b"biwkv_s", (2, 8, 0), (1, 9, -3)),
                            (b"biwkv_grid", (64, 0), (-1,)), (b"wkv6_fwd_scalar", (1, 0), (2, -1)),
                            (b"biwkv_bwd_serial", (1, 0), (5,))):
        for v in good:
            assert lib.vrwkv_set_option(name, v) == 0, (name, v)
            assert lib.vrwkv_get_option(name, ctypes.byref(val)) == 0 and val.value == v
        for v in bad:
            assert lib.vrwkv_set_option(name, v) == 1, (name, v)
            assert name in lib.vrwkv_last_error()
            assert lib.vrwkv_get_option(name, ctypes.byref(val)) == 0 and val.value == 0     # unchanged


def test_argument_validation_without_device(lib):
    f = lib.vrwkv_biwkv_fwd
    one = ctypes.c_void_p(16)
    # null pointers
    assert f(None, None, None, None, None, 1, 1, 1, 0, None, 0, None) == 1
    assert b"null" in lib.vrwkv_last_error()
    # non-positive sizes
    assert f(one, one, one, one, one, 0, 4, 4, 0, None, 0, None) == 1
    assert f(one, one, one, one, one, 1, -3, 4, 0, None, 0, None) == 1
    # unknown dtype code
    assert f(one, one, one, one, one, 1, 4, 4, 7, None, 0, None) == 2
    assert b"dtype" in lib.vrwkv_last_error()
    # misaligned tensor pointer
    assert f(one, one, ctypes.c_void_p(18), one, one, 1, 4, 4, 0, None, 0, None) == 1
    # a long sequence needs the workspace the query reports
    need = lib.vrwkv_biwkv_fwd_workspace_bytes(2, 4150, 768, 1)
    assert need > 0
    assert f(one, one, one, one, one, 2, 4150, 768, 1, None, 0, None) == 5
    assert b"workspace" in lib.vrwkv_last_error()
    assert lib.vrwkv_biwkv_fwd_workspace_bytes(64, 196, 768, 0) == 0
    # too large for 32-bit buffer offsets
    assert f(one, one, one, one, one, 1, 1 << 20, 1 << 10, 0, None, 0, None) == 3


def test_elementwise_entry_points_validate_without_device(lib):
    """The fused element-wise entry points reject bad arguments before touching the device."""
    one = ctypes.c_void_p(64)
    rf = lib.vrwkv_rowfuse
    assert rf(None, None, None, None, None, one, 4, 64, 0, 0, 1e-5, 1, None) == 1            # a is null
    assert rf(one, None, None, None, None, one, 4, 64, 0, 1, 1e-5, 1, None) == 1              # gate without `other`
    assert rf(one, None, one, None, None, one, 4, 64, 0, 0, 1e-5, 1, None) == 1               # LayerNorm weight without bias
    assert rf(one, None, None, None, None, one, 4, 60, 0, 0, 1e-5, 1, None) == 3              # N not a multiple of 8 (bf16)
    assert rf(one, None, None, None, None, one, 4, 64, 0, 0, 1e-5, 9, None) == 2              # unknown dtype
    assert rf(one, None, None, None, None, ctypes.c_void_p(72), 4, 64, 0, 0, 1e-5, 1, None) == 1   # misaligned output
    assert rf(one, None, None, None, None, one, 4, 64, 2, 0, 1e-5, 1, None) == 1              # unknown pre
    rb = lib.vrwkv_rowfuse_bwd
    assert lib.vrwkv_rowfuse_bwd_workspace_bytes(100, 768) == 25 * 3 * 768 * 4               # one partial row set per workgroup
    assert lib.vrwkv_rowfuse_bwd_workspace_bytes(1 << 20, 768) == 768 * 3 * 768 * 4         # ... of a grid of at most 768
    assert rb(one, one, None, None, None, one, one, None, None, 4, 64, 0, 1, 1e-5, 1, None, 0, None) == 1     # gate without gother
    assert rb(one, None, one, one, None, one, one, None, None, 4, 64, 0, 0, 1e-5, 1, None, 0, None) == 1      # LayerNorm without gparam
    assert rb(one, None, one, one, None, one, one, None, one, 4, 2048, 0, 0, 1e-5, 1, one, 1 << 20, None) == 3  # channel sums beyond 1024 channels
    assert rb(one, None, one, one, None, one, one, None, one, 4, 64, 0, 0, 1e-5, 1, None, 0, None) == 5       # workspace missing
    mm = lib.vrwkv_maa_mix
    outs = (ctypes.c_void_p * 5)(64, 64, 64, 64, 64)
    assert mm(one, one, one, one, outs, 0, 64, 1, None) == 1                                    # no rows
    assert mm(one, one, one, one, outs, 4, 60, 1, None) == 3                                    # C not a multiple of 8
    outs[3] = None
    assert mm(one, one, one, one, outs, 4, 64, 1, None) == 1                                    # a null output
    qb = lib.vrwkv_qshift_mix_bwd
    gp = (ctypes.c_void_p * 3)(64, 64, 64)
    need = lib.vrwkv_qshift_mix_bwd_workspace_bytes(3, 2, 196, 768)
    assert need == 2 * 7 * 3 * 768 * 4                                                        # one partial row per 32 tokens
    assert qb(one, one, gp, 3, one, one, 2, 196, 768, 14, 14, 1, 192, 0, 1, None, 0, None) == 5     # workspace missing
    assert b"workspace" in lib.vrwkv_last_error()
    assert qb(one, one, gp, 3, one, one, 2, 196, 768, 13, 14, 1, 192, 0, 1, one, need, None) == 3   # grid does not match T
    assert qb(one, one, gp, 4, one, one, 2, 196, 768, 14, 14, 1, 192, 0, 1, one, need, None) == 1   # n_mix out of range
    gp[1] = None
    assert qb(one, one, gp, 3, one, one, 2, 196, 768, 14, 14, 1, 192, 0, 1, one, need, None) == 1   # a null gradient
    gg = lib.vrwkv_groupnorm_gate
    assert gg(one, one, one, one, one, 4, 128, 64, 1e-5, 1, 0, None) == 2                      # fp32 gate beside a bf16 y
    assert gg(one, one, one, one, one, 4, 128, 48, 1e-5, 0, 1, None) == 3                      # C not a multiple of the group
    assert gg(one, one, one, one, one, 4, 96, 24, 1e-5, 0, 1, None) == 3                       # group not 8..128 in powers of two
    assert b"group" in lib.vrwkv_last_error()
    mb = lib.vrwkv_maa_mix_bwd
    gouts = (ctypes.c_void_p * 5)(64, 64, 64, 64, 64)
    assert lib.vrwkv_maa_mix_bwd_workspace_bytes(100, 768) == 4 * 5 * 768 * 4                 # one partial row set per 32 rows
    assert mb(one, one, one, one, gouts, one, one, one, None, 4, 64, 1, None, 0, None) == 1    # gmaa is null
    assert mb(one, one, one, one, gouts, one, one, one, one, 4, 64, 5, None, 0, None) == 2     # unknown dtype
    assert mb(one, one, one, one, gouts, one, one, one, one, 4, 60, 1, None, 0, None) == 3     # C not a multiple of 8
    assert mb(one, one, one, one, gouts, one, one, one, one, 4, 64, 1, None, 0, None) == 5     # workspace missing
    gouts[2] = None
    assert mb(one, one, one, one, gouts, one, one, one, one, 4, 64, 1, one, 1 << 20, None) == 1   # a null gradient
    gb = lib.vrwkv_groupnorm_gate_bwd
    assert lib.vrwkv_groupnorm_gate_bwd_workspace_bytes(100, 768) == 4 * 2 * 768 * 4          # one partial row pair per 32 rows
    assert gb(one, one, one, one, one, one, one, None, 4, 128, 64, 1e-5, 0, 1, None, 0, None) == 1    # gparam is null
    assert gb(one, one, one, one, one, one, one, one, 4, 128, 64, 1e-5, 2, 0, None, 0, None) == 2     # fp32 gate beside an fp16 y
    assert gb(one, one, one, one, one, one, one, one, 4, 2048, 64, 1e-5, 0, 1, None, 0, None) == 3    # more than 1024 channels
    assert gb(one, one, one, one, one, one, one, one, 4, 128, 64, 1e-5, 0, 1, None, 0, None) == 5     # workspace missing


def test_wkv6_backward_refuses_misaligned_pointers_without_device(lib):
    """Each tensor off its element size, and a workspace off 4 bytes, before anything is launched."""
    B, T, C, H = 1, 300, 64, 1
    for fn, like in ((lib.vrwkv_wkv6_bwd, False), (lib.vrwkv_wkv6_bwd_like, True)):
        for rkv, w in ((0, 0), (1, 0), (1, 1), (2, 2)):
            es, ws = (4 if rkv == 0 else 2), (4 if w == 0 else 2)
            out, outw = (es, ws) if like else (4, 4)
            #          r   k   v   w   u  gy gr   gk   gv   gw    gu workspace
            elements = [es, es, es, ws, 4, 4, out, out, out, outw, 4, 4]
            need = lib.vrwkv_wkv6_bwd_like_workspace_bytes(B, T, C, H, rkv, w) if like else lib.vrwkv_wkv6_bwd_workspace_bytes(B, T, C, H)
            for bad in range(len(elements)):
                p = [ctypes.c_void_p(4096 + (elements[i] // 2 if i == bad else 0)) for i in range(len(elements))]
                if fn(*[ctypes.cast(x, t) for x, t in zip(p[:11], fn.argtypes)], B, T, C, H, rkv, w, 0, p[11], need, None) != 1:
                    raise AssertionError((like, rkv, w, bad))
                assert b"aligned" in lib.vrwkv_last_error()


def test_block_entries_validate_without_device(lib):
    """vrwkv_block6_fwd takes a VRWKV6 block and all its parameters; null pointers and a short workspace are refused."""
    import vision_rwkv_amd as ops
    from vision_rwkv_amd import _lib
    B, T, C = 1, 12, 64
    size = lib.vrwkv_block_fwd_workspace_bytes(B, T, C, 256, 1, 1)
    names = ("ln1_w", "ln1_b", "ln2_w", "ln2_b", "key", "value", "receptance", "output", "ffn_key", "ffn_receptance", "ffn_value", "gate",
             "decay", "gn_w", "gn_b", "x", "out", "workspace")

    def call(missing=None, heads=1, bytes_=size, params=True):
        a = _lib.BlockArgs(B=B, T=T, C=C, hidden=256, heads=heads, Hp=3, Wp=4, shift_pixel=1, quarter=16, dtype=1, workspace_bytes=bytes_,
                           **{n: 4096 for n in names if n != missing})
        p = _lib.Block6Params(**{n: 4096 for n in _lib.Block6Params.POINTERS if n != missing})
        return lib.vrwkv_block6_fwd(ctypes.byref(a), ctypes.byref(p) if params else None, None)

    assert call(params=False) == 1 and call(heads=0) == 1
    for n in names + _lib.Block6Params.POINTERS[:13]:
        assert call(missing=n) == 1, n
    assert call(missing="att_kn_w") == 1                     # a norm's weight without its bias, and the other way round
    assert call(missing="att_kn_b") == 1
    assert call(bytes_=size - 1) == 5
    assert lib.vrwkv_block6_fwd(None, None, None) == 1 and lib.vrwkv_block_fwd(None, None) == 1


def test_linear_group_validates_without_device(lib):
    from vision_rwkv_amd import _lib

    def call(n=2, M=5, dtype=1, **change):
        f = dict(a=4096, w=4096, out=4096, N=32, K=64, lda=64, epi=0)
        return lib.vrwkv_linear_group((_lib.Linear * 2)(_lib.Linear(**f), _lib.Linear(**{**f, **change})), n, M, dtype, None)

    assert call(n=0) == 1 and call(n=6) == 1 and lib.vrwkv_linear_group(None, 1, 1, 1, None) == 1
    for name in ("a", "w", "out"):
        assert call(**{name: 0}) == 1 and call(**{name: 4104}) == 1
    for name in ("gate", "vec", "res"):
        assert call(**{name: 4104}) == 1
    assert call(epi=8) == 1
    refused = call(dtype=9)
    assert refused not in (0, 1)
    for change in (dict(M=0), dict(N=24), dict(K=48), dict(lda=56), dict(lda=68), dict(M=1 << 24), dict(N=1 << 23)):
        assert call(**change) not in (0, 1, refused), change


def test_more_sequences_than_a_grid_holds_are_not_cut(lib):
    """A forced number of segments does not apply to more sequences than the fold kernel's grid has rows."""
    import vision_rwkv_amd as ops
    with ops.option("wkv6_segments", 3):
        assert lib.vrwkv_wkv6_fwd_workspace_bytes(65535, 100, 64, 1) > 0
        assert lib.vrwkv_wkv6_fwd_workspace_bytes(65536, 100, 64, 1) == 0
        cut, uncut = (lib.vrwkv_wkv6_bwd_workspace_bytes(B, 100, 64, 1) / B for B in (65535, 65536))
    assert uncut == 201 * 64 * 4 and cut > 2 * 4 * 64 * 64 * 4         # two of two chunks each


def test_python_boundary_errors_without_device():
    import torch
    import vision_rwkv_amd as ops
    k = torch.randn(2, 8, 64)
    w = torch.zeros(64)
    with pytest.raises(RuntimeError, match="CUDA tensor"):
        ops.bi_wkv_forward(w, w, k, k)
    with pytest.raises(TypeError):
        ops.RUN_CUDA(w, w, k)


def test_bench_refuses_more_than_one_gpu_and_has_no_cpu_path():
    """bench.py runs on one GPU: --gpus 2 exits with a message instead of a number, and without a GPU the timed path
    refuses to run (nothing falls back to the CPU oracle)."""
    import subprocess
    import sys
    import torch
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert r.returncode != 0 and "one GPU" in r.stderr + r.stdout and "{" not in r.stdout
    if not torch.cuda.is_available():
        r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--steps", "1", "--warmup", "1"],
                           capture_output=True, text=True, timeout=300)
        assert r.returncode != 0 and "needs a GPU" in r.stderr and "{" not in r.stdout


def test_extension_module_stand_ins_and_torch_ops_namespaces():
    """The reference's three extension modules (bi_wkv.cpp:49-57, wkv_op.cpp:13-21, wkv6_op.cpp:13-21) have stand-ins
    with the same function names, also reachable through torch.ops."""
    import torch
    import vision_rwkv_amd as ops
    assert set(ops.ext.REGISTERED) == {"bi_wkv", "wkv", "wkv6"}
    for mod, names in ((ops.ext.bi_wkv, ("bi_wkv_forward", "bi_wkv_backward")), (ops.ext.wkv, ("forward", "backward")),
                       (ops.ext.wkv6, ("forward", "backward"))):
        for n in names:
            assert callable(getattr(mod, n))
    assert torch.ops.bi_wkv.bi_wkv_forward is not None and torch.ops.wkv.forward is not None
    assert torch.ops.wkv6.backward is not None
    k = torch.randn(2, 8, 64)
    with pytest.raises(RuntimeError, match="CUDA tensor"):
        ops.ext.wkv.forward(2, 8, 64, torch.zeros(64), torch.zeros(64), k, k, torch.empty_like(k))


@pytest.mark.parametrize("sequences,chunks", [(72, 9), (96, 10), (120, 10), (108, 11), (120, 13), (108, 14), (132, 19), (144, 24), (192, 130), (300, 130)])
def test_wkv6_sequences_that_are_faster_whole_are_not_cut(lib, sequences, chunks):
    """Shapes at which every count of segments measured slower than none, in any type (32-token chunks; 256 compute units): no workspace."""
    assert lib.vrwkv_wkv6_fwd_workspace_bytes(1, 32 * chunks, 64 * sequences, sequences) == 0


@pytest.mark.parametrize("sequences,chunks", [(1, 9), (3, 130), (12, 19), (48, 19), (36, 130), (84, 33), (96, 19)])
def test_wkv6_few_long_sequences_are_cut(lib, sequences, chunks):
    assert lib.vrwkv_wkv6_fwd_workspace_bytes(1, 32 * chunks, 64 * sequences, sequences) > 0


PARAM_VEC = r"""
#include "vrwkv_common.h"
#include <cstdlib>
#include <cstring>
int main() {
    for (int dtype : {VRWKV_F32, VRWKV_BF16, VRWKV_F16})
        for (int C : {1, 2, 3, 5, 8, 65}) {
            const int es = dtype == VRWKV_F32 ? 4 : 2;
            char* p = (char*)malloc((size_t)C * es);                  // ends where the vector ends
            for (int i = 0; i < C * es; ++i) p[i] = (char)(i + 1);
            const vrwkv::ParamVec v(p, dtype, 1.f);
            for (int c = 0; c < C; ++c) {
                unsigned want = 0;
                memcpy(&want, p + c * es, es);
                if (v.fetch(c) != want) return 1;
            }
            free(p);
        }
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_a_parameter_vector_is_read_element_by_element(tmp_path):
    """vrwkv_biwkv_fwd_as / _bwd_as ask for w and u aligned to their elements and for nothing around them: the fetch, compiled for the host under
    its address sanitizer, on vectors with nothing behind their last element."""
    (tmp_path / "v.hip").write_text(PARAM_VEC)
    csrc = os.path.join(ROOT, "vision-rwkv_amd", "csrc")
    build = "hipcc -O1 -std=c++17 --offload-arch=gfx950 --cuda-host-only -w -Xarch_host -fsanitize=address"
    subprocess.run([*build.split(), f"-I{csrc}", "-o", str(tmp_path / "v"), str(tmp_path / "v.hip")], check=True)
    done = subprocess.run([str(tmp_path / "v")], capture_output=True, text=True)
    assert done.returncode == 0, done.stderr[:2000]


@pytest.mark.parametrize("fault", ["missing", "another torch"])
def test_without_its_host_module_the_library_serves_the_python_classes(lib, fault, tmp_path, monkeypatch):
    """The compiled host side belongs to the torch that it was built with; the library does not, and used to serve the operators alone."""
    import torch
    from vision_rwkv_amd import _lib, ops
    monkeypatch.setattr(_lib, "_host", None)
    if fault == "missing":
        monkeypatch.setattr(_lib, "_HERE", str(tmp_path))
    else:
        monkeypatch.setattr(torch, "__version__", "1.0.0+other")
    with pytest.warns(RuntimeWarning, match="missing" if fault == "missing" else "built with torch"):
        host = _lib.host()
    assert host.wkv(1, 2, 3, 4, 1.0) is None and host.wkv6(*range(10)) is None and _lib.host() is host
    assert ops.block_weights_fit(torch.zeros(1, 1, 1), []) is False and ops.block_forward(torch.zeros(1, 1, 1), {}) is None
