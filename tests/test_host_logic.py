"""CPU-only tests: the oracle against the golden fixtures, the C-ABI library's exports and
argument validation (no kernel is launched), and the Python boundary's contract."""

from __future__ import annotations

import ctypes
import dataclasses
import hashlib
import pathlib
import re
import subprocess

import pytest
import torch

from oracle import naive_attention as oracle
from tests import golden_io

ROOT = pathlib.Path(__file__).resolve().parent.parent


# ------------------------------------------------------------------ oracle vs golden fixtures
@pytest.mark.parametrize("name", golden_io.NAMES)
def test_oracle_reproduces_golden_fixture(name):
    g = golden_io.load(name)
    o, dq, dk, dv = oracle.naive_backward(g["q"], g["k"], g["v"], g["d_o"], g["scale"], torch.float32)
    lse = oracle.naive_lse(g["q"], g["k"], g["scale"])
    for got, key in ((o, "o"), (dq, "dq"), (dk, "dk"), (dv, "dv"), (lse, "lse")):
        torch.testing.assert_close(got, g[key], atol=2e-5, rtol=2e-5)


# ------------------------------------------------------------------ C ABI: exports and errors
def _declared_functions() -> list[str]:
    text = (ROOT / "include" / "fa2_gfx950.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return re.findall(r"\b(fa2_[a-z0-9_]+)\s*\(", text)


def test_library_exports_every_declared_symbol(capi):
    lib = capi.load()
    names = sorted(set(_declared_functions()))
    assert names, "no declarations found in include/fa2_gfx950.h"
    for name in names:
        assert hasattr(lib, name), f"libfa2_gfx950.so does not export {name}"
    assert sorted(capi.SIGNATURES) == names, "ctypes binding and header disagree on the entry points"


# sha256 (first 16 digits) of include/fa2_gfx950.h without comments, white space and the version itself, per ABI
# version.  A change of the interface needs a new version and a line here.
INTERFACES = {6: "94837833e0c9a376", 7: "f98a87f9170d5460", 8: "6532f24f44a70406", 9: "1aebc81505efa417"}


def test_abi_version_follows_the_interface(capi):
    text = re.sub(r"/\*.*?\*/", " ", (ROOT / "include" / "fa2_gfx950.h").read_text(), flags=re.S)
    version = int(re.search(r"#define FA2_ABI_VERSION (\d+)", text).group(1))
    text = " ".join(re.sub(r"#define FA2_ABI_VERSION \d+", "", text).split())
    assert version == capi.ABI_VERSION == max(INTERFACES)
    assert hashlib.sha256(text.encode()).hexdigest()[:16] == INTERFACES[version]


def test_library_of_another_version_is_refused_by_name(capi, tmp_path, monkeypatch):
    """Also one that lacks entry points of this version: the error says which version it has, not which symbol."""
    (tmp_path / "old.c").write_text("int fa2_abi_version(void) { return 5; }\n")
    old = tmp_path / "libfa2_gfx950.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(old), str(tmp_path / "old.c")], check=True)
    monkeypatch.setattr(capi, "LIBRARY_PATH", old)
    monkeypatch.setattr(capi, "_lib", None)
    with pytest.raises(RuntimeError, match="ABI version 5, binding expects"):
        capi.load()


def test_abi_version_and_table(capi):
    lib = capi.load()
    assert lib.fa2_abi_version() == capi.ABI_VERSION
    rows = capi.config_table()
    assert [r["id"] for r in rows] == list(range(len(rows)))
    # The rows FA2_CONFIG_AUTO picks from (plain), and the forward-only rows whose forward folds the
    # softmax scale into Q (what fa2_pick_config_forward_only returns for bf16 up to 128 columns).
    plain = [r for r in rows if not r["dq_atomic"] and not r["fwd_exp_folded"]]
    folded = [r for r in rows if r["fwd_exp_folded"]]
    assert [r["headdim_padded"] for r in plain] == [32, 64, 96, 128, 192, 256]
    assert [r["headdim_padded"] for r in folded] == [32, 64, 96, 128]
    assert plain[-1]["headdim_padded"] == capi.FA2_MAX_HEADDIM
    for r in rows:
        assert r["fwd_block_q"] == 32 * r["fwd_waves"]
        assert r["bwd_block_kv"] == 32 * r["bwd_waves"]
        assert r["dq_block_q"] == 32 * r["dq_waves"]
    by_dim = {r["headdim_padded"]: r for r in plain}
    for r in folded:  # a folded row differs from the plain row of its head dimension in that flag only
        twin = dict(by_dim[r["headdim_padded"]], id=r["id"], fwd_exp_folded=1)
        assert r == twin and not r["dq_atomic"]
    for d, want in ((1, 32), (32, 32), (33, 64), (48, 64), (64, 64), (96, 96), (100, 128), (128, 128),
                    (129, 192), (192, 192), (193, 256), (256, 256)):
        for dtype, seqlen in ((capi.FA2_DTYPE_F16, 512), (capi.FA2_DTYPE_BF16, 512), (capi.FA2_DTYPE_BF16, 16384)):
            idx = lib.fa2_pick_config(dtype, d, seqlen, seqlen, 0)
            assert idx >= 0 and rows[idx]["headdim_padded"] == want
            assert not rows[idx]["dq_atomic"] and not rows[idx]["fwd_exp_folded"]
            assert lib.fa2_pick_config(dtype, d, seqlen, seqlen, 1) == idx  # both backward modes share the row
            only = lib.fa2_pick_config_forward_only(dtype, d, seqlen, seqlen)
            assert only >= 0 and rows[only]["headdim_padded"] == want and not rows[only]["dq_atomic"]
            assert rows[only]["fwd_exp_folded"] == int(dtype == capi.FA2_DTYPE_BF16 and want <= 128)
    assert lib.fa2_pick_config_forward_only(capi.FA2_DTYPE_BF16, 257, 512, 512) == -4  # FA2_ERR_HEADDIM
    # LDS-direct kernels: all three up to 128 columns, forward and dQ only at 192 and 256.
    assert [r["lds_direct"] for r in plain] == [1, 1, 1, 1, 2, 2]
    # (batch, head) pairs dispatched together: a multiple of 8 (one XCD per head), fewer at 128 columns.
    assert all(r["head_group"] % 8 == 0 and r["head_group"] > 0 for r in rows)
    assert by_dim[128]["head_group"] < by_dim[64]["head_group"]
    assert lib.fa2_pick_config(capi.FA2_DTYPE_BF16, 257, 512, 512, 0) == -4  # FA2_ERR_HEADDIM
    assert lib.fa2_pick_config(7, 64, 512, 512, 0) == -3  # FA2_ERR_BAD_DTYPE
    info = capi.ConfigInfo()
    assert lib.fa2_config_get(99, ctypes.byref(info)) == 6  # FA2_ERR_BAD_CONFIG
    assert lib.fa2_config_get(0, None) == 1  # FA2_ERR_NULL_POINTER


def _fwd_args(capi, **over):
    a = dict(q=16, k=16, v=16, o=16, lse=16, batch=1, nheads=1, seqlen_q=8, seqlen_k=8, headdim=64,
             seqlen_q_rounded=128, scale=0.125, dtype=capi.FA2_DTYPE_F16, config=capi.FA2_CONFIG_AUTO)
    a.update(over)
    strides = [a["seqlen_q"] * a["headdim"], a["seqlen_q"] * a["headdim"], a["headdim"]] * 4
    if "strides" in over:
        strides = over["strides"]
    return [a["q"], a["k"], a["v"], a["o"], a["lse"], a["batch"], a["nheads"], a["seqlen_q"], a["seqlen_k"],
            a["headdim"], a["seqlen_q_rounded"], *strides, a["scale"], a["dtype"], a["config"], None]


@pytest.mark.parametrize("over,status", [
    (dict(q=None), "FA2_ERR_NULL_POINTER"),
    (dict(lse=None), "FA2_ERR_NULL_POINTER"),
    (dict(batch=0), "FA2_ERR_BAD_SHAPE"),
    (dict(seqlen_k=-3), "FA2_ERR_BAD_SHAPE"),
    (dict(seqlen_q=300, seqlen_q_rounded=256), "FA2_ERR_BAD_SHAPE"),
    (dict(headdim=264), "FA2_ERR_HEADDIM"),
    (dict(dtype=5), "FA2_ERR_BAD_DTYPE"),
    (dict(config=17), "FA2_ERR_BAD_CONFIG"),
    (dict(config=0, headdim=64), "FA2_ERR_BAD_CONFIG"),  # row 0 is built for headdim <= 32
    (dict(scale=float("nan")), "FA2_ERR_BAD_SHAPE"),
    (dict(strides=[-1] * 12), "FA2_ERR_BAD_STRIDE"),
])
def test_forward_rejects_bad_arguments_before_launching(capi, over, status):
    """Every error returns a status and a message; nothing is launched, thrown or aborted."""
    lib = capi.load()
    rc = lib.fa2_fwd(*_fwd_args(capi, **over))
    assert rc != 0
    assert lib.fa2_status_string(rc).decode() == status
    assert lib.fa2_last_error_string().decode() != ""
    with pytest.raises(RuntimeError, match=status):
        capi.check(rc, "fa2_fwd")


def test_backward_entry_points_reject_bad_arguments(capi):
    lib = capi.load()
    st = [512, 512, 64]
    rc = lib.fa2_bwd_preprocess(None, 16, 16, 1, 1, 8, 64, 128, *st, *st, capi.FA2_DTYPE_F16, None)
    assert lib.fa2_status_string(rc).decode() == "FA2_ERR_NULL_POINTER"
    rc = lib.fa2_bwd_preprocess(16, 16, 16, 1, 1, 8, 300, 128, *st, *st, capi.FA2_DTYPE_F16, None)
    assert lib.fa2_status_string(rc).decode() == "FA2_ERR_HEADDIM"
    rc = lib.fa2_bwd(16, 16, 16, 16, 16, None, None, 16, 16, 16, 1, 1, 8, 8, 64, 128, *(st * 7),
                     0.125, capi.FA2_DTYPE_F16, 1, capi.FA2_CONFIG_AUTO, None)
    assert lib.fa2_status_string(rc).decode() == "FA2_ERR_NULL_POINTER"
    assert "delta" in lib.fa2_last_error_string().decode()
    rc = lib.fa2_bwd(16, 16, 16, 16, 16, 16, None, 16, 16, 16, 1, 1, 0, 8, 64, 128, *(st * 7),
                     0.125, capi.FA2_DTYPE_F16, 1, capi.FA2_CONFIG_AUTO, None)
    assert lib.fa2_status_string(rc).decode() == "FA2_ERR_BAD_SHAPE"
    assert lib.fa2_bwd_workspace_bytes(2, 4, 512, 512, 64, 1, capi.FA2_CONFIG_AUTO) == 0
    # Either gradient group may be omitted, but not both, and dk/dv only together.
    rc = lib.fa2_bwd(16, 16, 16, 16, 16, 16, None, None, None, None, 1, 1, 8, 8, 64, 128, *(st * 7),
                     0.125, capi.FA2_DTYPE_F16, 1, capi.FA2_CONFIG_AUTO, None)
    assert lib.fa2_status_string(rc).decode() == "FA2_ERR_NULL_POINTER"
    assert "all NULL" in lib.fa2_last_error_string().decode()
    rc = lib.fa2_bwd(16, 16, 16, 16, 16, 16, None, 16, 16, None, 1, 1, 8, 8, 64, 128, *(st * 7),
                     0.125, capi.FA2_DTYPE_F16, 1, capi.FA2_CONFIG_AUTO, None)
    assert lib.fa2_status_string(rc).decode() == "FA2_ERR_NULL_POINTER"
    assert "dv" in lib.fa2_last_error_string().decode()
    # A forward-only row (its forward rounds Q * scale) is refused by the backward.
    only = lib.fa2_pick_config_forward_only(capi.FA2_DTYPE_BF16, 64, 8, 8)
    assert capi.config_table()[only]["fwd_exp_folded"] == 1
    rc = lib.fa2_bwd(16, 16, 16, 16, 16, 16, None, 16, 16, 16, 1, 1, 8, 8, 64, 128, *(st * 7),
                     0.125, capi.FA2_DTYPE_BF16, 1, only, None)
    assert lib.fa2_status_string(rc).decode() == "FA2_ERR_BAD_CONFIG"
    assert "forward-only" in lib.fa2_last_error_string().decode()


def test_fp32_entry_points_reject_bad_arguments(capi):
    """fa2_fwd_packed_f32_out and fa2_cast_f32_to_f16: every refusal comes before anything is launched."""
    lib = capi.load()

    def fwd(o_f32, o=16, args=True):
        t = capi.Tensor(16, 512, 512, 64)
        a = capi.FwdArgs(t, t, t, capi.Tensor(o, 512, 512, 64), 16, 1, 1, 0, 8, 64, 128, 0.125, capi.FA2_DTYPE_F16,
                         capi.FA2_CONFIG_AUTO)
        return lib.fa2_status_string(lib.fa2_fwd_packed_f32_out(ctypes.byref(a) if args else None, o_f32, None)).decode()

    assert fwd(16, args=False) == fwd(None) == "FA2_ERR_NULL_POINTER"
    assert fwd(18) == "FA2_ERR_BAD_STRIDE"
    assert fwd(20) == fwd(16, o=None) == "FA2_ERR_BAD_SHAPE"  # seqlen_q is 0; the pointers are fine
    t = capi.Tensor(16, 512, 512, 64)
    a = capi.FwdArgs(t, t, t, capi.Tensor(None, 0, 0, 0), 16, 1, 1, 8, 8, 64, 128, 0.125, capi.FA2_DTYPE_F16, capi.FA2_CONFIG_AUTO)
    assert lib.fa2_status_string(lib.fa2_fwd_packed(ctypes.byref(a), None)).decode() == "FA2_ERR_NULL_POINTER"

    def cast(*jobs, count=None):
        arrays = (capi.Cast * max(1, len(jobs)))(*(capi.Cast(*j) for j in jobs))
        n = len(jobs) if count is None else count
        return lib.fa2_status_string(lib.fa2_cast_f32_to_f16(arrays if jobs else None, n, None)).decode()

    good = (16, 16, 8)
    assert cast(count=1) == "FA2_ERR_NULL_POINTER"
    assert cast(good, count=0) == cast(good, count=4) == "FA2_ERR_BAD_SHAPE"
    assert cast(good, (None, 16, 8)) == cast((16, None, 8)) == "FA2_ERR_NULL_POINTER"
    assert cast((16, 16, 0)) == cast(good, good, (16, 16, -1)) == "FA2_ERR_BAD_SHAPE"
    assert cast((24, 16, 8)) == cast((16, 20, 8)) == "FA2_ERR_BAD_STRIDE"
    assert cast(good, (16, 16, 1 << 60)) == cast(*[(16, 16, 1 << 35)] * 3) == "FA2_ERR_TOO_LARGE"


def test_missing_library_fails_loudly(capi, monkeypatch, tmp_path):
    monkeypatch.setattr(capi, "_lib", None)
    monkeypatch.setattr(capi, "LIBRARY_PATH", tmp_path / "libfa2_gfx950.so")
    with pytest.raises(RuntimeError, match="not built"):
        capi.load()


# ------------------------------------------------------------------ Python boundary contract
def test_public_names_match_reference(fa):
    """Reference: src/flash_attention_triton/__init__.py:13."""
    for name in ("KernelsConfigV2", "flash_attention_v2", "flash_attention_v2_custom", "init_to_zero_v2"):
        assert name in fa.__all__ and hasattr(fa, name)


def test_kernels_config_is_a_frozen_record_with_reference_fields(fa):
    fields = [f.name for f in dataclasses.fields(fa.KernelsConfigV2)]
    # The reference's nine fields in its order (_configurators_v2.py:27-38), then the one optional
    # field this package adds; a configuration written for the reference constructs unchanged.
    assert fields == ["block_rows_size", "block_cols_size", "min_block_headdim", "max_headdim",
                      "seqlen_cache_divisor", "min_warps", "max_warps", "num_stages",
                      "backward_autotune_configs", "exact_scale"]
    cfg = fa.KernelsConfigV2(128, 64, 32, 128, 32, 4, 4, 2, [
        fa.BackwardConfig({"BLOCK_Q_ROWS_SIZE": 64, "BLOCK_KV_COLS_SIZE": 128, "SEQUENCE_PARALLEL": False},
                          num_warps=4, num_stages=2, pre_hook=fa.init_to_zero_v2("DQ"))])
    with pytest.raises(dataclasses.FrozenInstanceError):
        cfg.block_rows_size = 64
    assert cfg.deterministic is True and cfg.exact_scale is False
    par = dataclasses.replace(cfg, backward_autotune_configs=[
        fa.BackwardConfig({"BLOCK_Q_ROWS_SIZE": 64, "BLOCK_KV_COLS_SIZE": 128, "SEQUENCE_PARALLEL": True})])
    assert par.deterministic is False


def test_init_to_zero_hook_zeroes_named_tensor(fa):
    hook = fa.init_to_zero_v2("DQ")
    t = torch.ones(4)
    assert hook({"DQ": t, "DK": torch.ones(2)}) is t
    assert torch.count_nonzero(t) == 0


def test_selector_and_validation(fa2_module, monkeypatch):
    sel = fa2_module._select_optimal_gpu_architecture
    assert sel((9, 5), True) is fa2_module.GFX950_KERNEL_CONFIG_DETERMINISTIC
    assert sel((9, 5), False) is fa2_module.GFX950_KERNEL_CONFIG_NON_DETERMINISTIC
    assert sel((9, 5), True).deterministic and not sel((9, 5), False).deterministic
    with pytest.raises(ValueError, match="Unsupported GPU compute capability"):
        sel((9, 4), False)
    with pytest.raises(RuntimeError, match="gfx950"):
        fa2_module._validate_runtime_compatibility((9, 4), "gfx942:sramecc+:xnack-")
    fa2_module._validate_runtime_compatibility((9, 5), "gfx950:sramecc+:xnack-")

    # flash_attention_v2_custom: a missing key for the current device is a ValueError
    monkeypatch.setattr(torch.cuda, "get_device_capability", lambda *a, **k: (9, 5))
    q = torch.zeros(1, 1, 4, 8)
    with pytest.raises(ValueError, match="Missing kernel configuration"):
        fa2_module.flash_attention_v2_custom(q, q, q, None, {(8, 0): sel((9, 5), True)})


def test_custom_tile_fields_are_reported_not_silently_dropped(fa, fa2_module, monkeypatch):
    """The reference passes a custom configuration's tile and warp values to its kernels
    (flash_attention_2.py:137-141); here they cannot change the compiled kernels, and the caller is
    told so once.  The compiled shapes themselves raise no warning."""
    import warnings

    monkeypatch.setattr(fa2_module, "_TILE_WARNING_SHOWN", False)
    ampere = fa.KernelsConfigV2(256, 256, 32, 256, 32, 8, 8, 1, [
        fa.BackwardConfig({"BLOCK_Q_ROWS_SIZE": 128, "BLOCK_KV_COLS_SIZE": 128, "SEQUENCE_PARALLEL": False})])
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        fa2_module._warn_about_ignored_tile_fields(fa2_module.GFX950_KERNEL_CONFIG_DETERMINISTIC)
        fa2_module._warn_about_ignored_tile_fields(fa2_module.GFX950_KERNEL_CONFIG_SEQUENCE_PARALLEL_ATOMIC)
        assert not seen
        fa2_module._warn_about_ignored_tile_fields(ampere)
        fa2_module._warn_about_ignored_tile_fields(ampere)
    assert len(seen) == 1 and "ignored" in str(seen[0].message) and "exact_scale" in str(seen[0].message)


def test_launcher_assertions_mirror_reference(fa2_module):
    """Same AssertionErrors as flash_attention_2.py:85-90, raised before any FFI call."""
    cfg = fa2_module.GFX950_KERNEL_CONFIG_DETERMINISTIC
    tail = (cfg.block_rows_size, cfg.block_cols_size, cfg.min_block_headdim, cfg.max_headdim,
            cfg.seqlen_cache_divisor, cfg.min_warps, cfg.max_warps, cfg.num_stages)
    fwd = fa2_module._flash_attention_forward
    q = torch.zeros(1, 2, 8, 16, dtype=torch.float16)
    with pytest.raises(AssertionError):
        fwd(q, torch.zeros(1, 2, 8, 32, dtype=torch.float16), q, None, *tail)  # k shape
    with pytest.raises(AssertionError):
        fwd(q, q, torch.zeros(1, 3, 8, 16, dtype=torch.float16), None, *tail)  # v shape
    big = torch.zeros(1, 1, 4, 264, dtype=torch.float16)
    with pytest.raises(AssertionError, match="Supports head dimensions only up to 256"):
        fwd(big, big, big, None, *tail)
    with pytest.raises(AssertionError, match="must reside on CUDA device"):
        fwd(q, q, q, None, *tail)


def test_backward_record_follows_the_lse_row_length(fa2_module, monkeypatch):
    """The cached argument record of the backward launcher is per padded lse row length: the same
    shapes under another max_headdim (N = 100 pads to 256 or to 128, flash_attention_2.py:98) must
    not be handed the earlier call's seqlen_q_rounded, which the kernels index lse and delta with."""
    seen = []

    class FakeLibrary:
        @staticmethod
        def fa2_bwd_workspace_bytes(*_):
            return 0

        @staticmethod
        def fa2_bwd_packed(args, _stream):
            seen.append((args.seqlen_q, args.seqlen_q_rounded))
            return 0

    monkeypatch.setattr(fa2_module._capi, "load", lambda: FakeLibrary)
    monkeypatch.setattr(fa2_module, "_stream_handle", lambda: 0)
    base = fa2_module.GFX950_KERNEL_CONFIG_DETERMINISTIC
    q = torch.zeros(1, 2, 100, 64, dtype=torch.float16)
    grads = [torch.empty_like(q) for _ in range(3)]
    for max_headdim, rounded in ((256, 256), (128, 128), (256, 256)):
        cfg = dataclasses.replace(base, max_headdim=max_headdim)
        lse = torch.zeros(1, 2, rounded)
        fa2_module._flash_attention_backward(q, q, q, q, lse, *grads, q, None, cfg)
        with pytest.raises(AssertionError):  # an lse of another row length is refused, as in the reference
            fa2_module._flash_attention_backward(q, q, q, q, torch.zeros(1, 2, rounded + 128), *grads, q, None, cfg)
    assert seen == [(100, 256), (100, 128), (100, 256)]


def test_cpp_autograd_node_is_built_and_matches_the_library(capi, fa2_module):
    """The C++ autograd node (csrc/fa2_torch_autograd.cpp) loads without a GPU, is linked against
    the same ABI as the ctypes binding, and is what the public functions record."""
    node = fa2_module._cpp_node()
    assert node is not None, "flash-attention-triton_amd/_fa2_torch.so is not built (python flash-attention-triton_amd/build.py)"
    assert node.abi_version() == capi.ABI_VERSION
    q = torch.zeros(1, 2, 8, 16, dtype=torch.float16)
    with pytest.raises(AssertionError, match="must reside on CUDA device"):  # the launcher's checks come first
        fa2_module._apply(q, q, q, None, fa2_module.GFX950_KERNEL_CONFIG_DETERMINISTIC)


def test_grids_beyond_a_launch_are_refused(capi):
    """Of a grid of 2^32 threads and more only the remainder modulo 2^32 would run, silently: the entry points
    refuse it before anything touches a device."""
    lib = capi.load()
    heads = 2**24  # 256 threads each
    t = capi.Tensor(16, 0, 0, 0)
    fwd = capi.FwdArgs(q=t, k=t, v=t, o=t, lse=16, batch=heads, nheads=1, seqlen_q=1, seqlen_k=1, headdim=8,
                       seqlen_q_rounded=1, softmax_scale=1.0, dtype=capi.FA2_DTYPE_F16, config_id=capi.FA2_CONFIG_AUTO)
    assert lib.fa2_status_string(lib.fa2_fwd_packed(fwd, None)) == b"FA2_ERR_TOO_LARGE"
    bwd = capi.BwdArgs(q=t, k=t, v=t, o=t, d_o=t, dq=t, dk=t, dv=t, lse=16, delta=16, batch=heads, nheads=1, seqlen_q=1,
                       seqlen_k=1, headdim=8, seqlen_q_rounded=1, softmax_scale=1.0, dtype=capi.FA2_DTYPE_F16,
                       config_id=capi.FA2_CONFIG_AUTO)
    assert lib.fa2_status_string(lib.fa2_bwd_packed(bwd, None)) == b"FA2_ERR_TOO_LARGE"


def test_noalloc_entry_point_refuses_sizes_beyond_its_scratch(capi):
    """The size check of fa2_bwd_fused_noalloc comes before anything touches a device."""
    lib = capi.load()
    n_r = 1024
    b = capi.FA2_NOALLOC_MAX_ROWS // n_r + 1
    args = [16] * 9 + [b, 1, n_r, n_r, 64, n_r] + [0] * 24 + [0.125, capi.FA2_DTYPE_F16, 0, capi.FA2_CONFIG_AUTO, None]
    status = lib.fa2_bwd_fused_noalloc(*args)
    assert lib.fa2_status_string(status) == b"FA2_ERR_TOO_LARGE"
    assert b"FA2_NOALLOC_MAX_ROWS" in lib.fa2_last_error_string()


def test_sequence_parallel_rows_and_workspace(capi, fa2_module):
    """The table's sequence-parallel rows are never picked automatically, size their workspace, and
    the configuration classes select them."""
    lib = capi.load()
    rows = capi.config_table()
    atomic = [r for r in rows if r["dq_atomic"]]
    assert sorted(r["headdim_padded"] for r in atomic) == [32, 64, 128]
    for d in (8, 32, 64, 96, 128, 200, 256):
        assert rows[lib.fa2_pick_config(capi.FA2_DTYPE_BF16, d, 512, 512, 0)]["dq_atomic"] == 0
    for r in atomic:
        d = r["headdim_padded"]
        assert lib.fa2_bwd_workspace_bytes(2, 3, 130, 77, d, 0, r["id"]) == 2 * 3 * 192 * d * 4
        assert lib.fa2_bwd_workspace_bytes(2, 3, 130, 77, d, 0, capi.FA2_CONFIG_AUTO) == 0
    assert fa2_module.GFX950_KERNEL_CONFIG_SEQUENCE_PARALLEL_ATOMIC.atomic_dq
    assert not fa2_module.GFX950_KERNEL_CONFIG_SEQUENCE_PARALLEL_ATOMIC.deterministic
    assert not fa2_module.GFX950_KERNEL_CONFIG_NON_DETERMINISTIC.atomic_dq
    assert not fa2_module.GFX950_KERNEL_CONFIG_DETERMINISTIC.atomic_dq


def test_workload_table_matches_baseline(workloads):
    w = workloads.WORKLOADS
    assert w["C1"].shape == (2, 4, 512, 64) and w["C1"].dtype == torch.float16
    assert w["C2"].shape == (4, 16, 2048, 64) and w["C2"].dtype == torch.bfloat16 and w["C2"].both_modes
    assert w["C3"].shape == (2, 32, 4096, 128) and w["C3"].dtype == torch.bfloat16
    assert w["C4"].shape == (1, 16, 16384, 128) and w["C4"].both_modes
    assert w["C5"].shape == (8, 12, 3000, 64) and w["C5"].qk_std == 3.0
    assert w["C3"].fwd_flops == pytest.approx(274.88e9, rel=1e-3)
    assert w["C3"].fwd_bytes == pytest.approx(269.5e6, rel=1e-3)
    q, k, v, g = workloads.make_inputs(w["C1"])
    q2, *_ = workloads.make_inputs(w["C1"], heads=3)
    assert q.dtype == torch.float16 and q.shape == (2, 4, 512, 64)
    torch.testing.assert_close(q2[:, 0], q.reshape(8, 512, 64)[:3], atol=0, rtol=0)


def test_launch_info_says_what_a_call_launches(capi, workloads):
    """fa2_launch_info_get against tiles and grids written out here, and the kernel names the bench derives from it."""
    import importlib

    bench = importlib.import_module("bench")
    rows = capi.config_table()

    def part(form, block_rows, key_groups, wg_per_cu, resident, workgroups):
        return dict(form=form, block_rows=block_rows, key_groups=key_groups, wg_per_cu=wg_per_cu, resident=resident,
                    workgroups=workgroups)

    info = capi.launch_info(2, 32, 4096, 4096, 128)
    assert info == {"config_id": 3, "fwd": part("direct", 128, 1, 2, 0, 2048), "dq": part("direct", 128, 1, 2, 0, 2048),
                    "dkdv": part("paired", 64, 1, 2, 0, 4096)}
    assert [bench.kernel_name(info, p) for p in ("fwd", "dq", "dkdv")] == [
        "fwd_direct_kernel", "bwd_dq_direct_kernel", "bwd_dkdv_pair_kernel"]
    info = capi.launch_info(1, 16, 16384, 16384, 128)  # longer than the paired kernel pays
    assert info["dkdv"] == part("direct", 128, 1, 1, 0, 2048)
    assert bench.kernel_name(info, "dkdv") == "bwd_dkdv_direct_kernel"
    info = capi.launch_info(2, 4, 512, 512, 64)  # 32 workgroups of 128 rows for 256 CUs: two key groups
    assert info["fwd"] == info["dq"] == part("direct", 64, 2, 3, 1, 64)
    assert info["dkdv"] == part("paired", 64, 1, 3, 1, 64)
    assert capi.launch_info(32, 20, 1024, 1024, 96)["dkdv"] == part("paired", 64, 1, 2, 0, 10240)
    info = capi.launch_info(2, 8, 100, 200, 50)  # 50 columns: no 16-byte rows
    assert info["fwd"] == info["dq"] == part("generic", 128, 1, 0, 0, 16)
    assert info["dkdv"] == part("generic", 128, 1, 0, 0, 32)
    assert [bench.kernel_name(info, p) for p in ("fwd", "dq", "dkdv")] == ["fwd_kernel", "bwd_dq_kernel", "bwd_dkdv_kernel"]
    atomic = next(r for r in rows if r["dq_atomic"] and r["headdim_padded"] == 128)
    info = capi.launch_info(2, 32, 4096, 4096, 128, atomic["id"])
    assert info["dkdv"] == part("direct", 128, 1, atomic["dkdv_wg_per_cu"], 0, 2048) and not any(
        v for k, v in info["dq"].items() if k != "form")
    folded = next(r for r in rows if r["fwd_exp_folded"] and r["headdim_padded"] == 128)
    info = capi.launch_info(2, 32, 4096, 4096, 128, folded["id"])
    assert info["fwd"]["form"] == "direct" and info["dkdv"]["workgroups"] == info["dq"]["workgroups"] == 0
    with pytest.raises(RuntimeError, match="FA2_ERR_BAD_SHAPE"):
        capi.launch_info(0, 1, 1, 1, 64)
    with pytest.raises(RuntimeError, match="FA2_ERR_BAD_CONFIG"):
        capi.launch_info(1, 1, 1, 1, 64, 99)


def test_launch_info_knows_grids_of_two_kinds(capi):
    """The forward that mixes one and two key groups, and the backward's joint grid: its runs of 8 workgroups, of which every third
    (two key groups: every second) is of dQ, cover both kinds."""
    import importlib

    bench = importlib.import_module("bench")
    for config in (capi.FA2_CONFIG_AUTO, capi.load().fa2_pick_config_forward_only(capi.FA2_DTYPE_BF16, 128, 4096, 4096)):
        info = capi.launch_info(1, 16, 4096, 4096, 128, config)  # 64 tiles of 64 rows per head: 24 pairs and 16 by themselves
        assert info["fwd"] == dict(form="mixed", block_rows=128, key_groups=1, wg_per_cu=2, resident=0, workgroups=16 * 40)
        assert bench.kernel_name(info, "fwd") == "fwd_mixed_kernel"
    assert capi.launch_info(1, 16, 4095, 4095, 128)["fwd"]["form"] == "direct"
    part = dict(form="joint", block_rows=64, key_groups=2, wg_per_cu=3, resident=1, workgroups=128)
    assert capi.joint_info(2, 4, 512, 512, 64) == part  # 64 workgroups of 64 rows and 64 of 64 keys
    assert capi.joint_info(1, 32, 2048, 2048, 64) == {**part, "block_rows": 128, "key_groups": 1, "resident": 0, "workgroups": 3 * 512}
    assert capi.joint_info(1, 8, 4096, 4096, 128) == {**part, "block_rows": 128, "key_groups": 1, "wg_per_cu": 2, "resident": 0, "workgroups": 768}
    assert capi.launch_info(1, 8, 4096, 4096, 128)["dq"]["key_groups"] == 2  # in front of a dK/dV kernel; two launches are not what runs
    for sizes in [(2, 32, 4096, 4096, 128), (2, 4, 512, 2049, 64), (1, 8, 100, 100, 50)]:  # large; longer keys; no 16-byte rows
        assert capi.joint_info(*sizes) is None
    for row in capi.config_table():
        if row["headdim_padded"] == 64 and (row["dq_atomic"] or row["fwd_exp_folded"]):
            assert capi.joint_info(2, 4, 512, 512, 64, row["id"]) is None
    with pytest.raises(RuntimeError, match="FA2_ERR_BAD_SHAPE"):
        capi.joint_info(0, 1, 1, 1, 64)


@pytest.mark.parametrize("heads,n,d,fwd,dq", [
    (60, 64, 128, 1, 1), (60, 65, 128, 2, 2), (8, 65, 256, 2, 1), (8, 97, 256, 2, 2),  # at most 128 workgroups of 128 rows
    (128, 256, 32, 2, 2), (77, 333, 64, 2, 1), (128, 256, 64, 2, 2), (59, 333, 96, 2, 1), (77, 384, 96, 1, 1), (58, 512, 96, 2, 2),  # 256
    (72, 256, 128, 2, 1), (116, 256, 128, 1, 1), (59, 384, 128, 1, 1), (51, 512, 128, 1, 1), (64, 512, 128, 2, 2),
    (33, 500, 128, 2, 2), (47, 640, 128, 1, 1), (29, 1024, 128, 2, 2), (29, 1024, 256, 1, 1), (32, 1024, 256, 2, 2), (17, 1024, 192, 2, 2), (15, 2048, 192, 2, 2),
    (75, 512, 32, 2, 2), (75, 512, 64, 1, 1), (96, 512, 64, 2, 2), (43, 1024, 64, 2, 2), (24, 2048, 96, 2, 2),  # 384
    (24, 2048, 128, 1, 1), (12, 4096, 128, 2, 2), (10, 4096, 256, 1, 1),
    (64, 1024, 32, 2, 2), (16, 4096, 64, 2, 2), (64, 1024, 64, 1, 1), (16, 4096, 128, 1, 1), (17, 4096, 32, 1, 1)])  # 512
def test_two_key_groups_only_where_they_measured_faster(capi, heads, n, d, fwd, dq):
    """The forward's and dQ's key groups on both sides of every line of the rule."""
    info = capi.launch_info(1, heads, n, n, d)
    assert (info["fwd"]["key_groups"], info["dq"]["key_groups"]) == (fwd, dq)


@pytest.mark.parametrize("heads,n,d,fwd,dq", [
    (59, 333, 48, 2, 2), (63, 500, 48, 2, 2), (65, 255, 40, 1, 1), (59, 333, 64, 2, 1), (70, 300, 64, 2, 2),
    (63, 500, 56, 2, 1), (63, 512, 64, 2, 2), (59, 333, 80, 2, 2), (61, 333, 72, 2, 2), (67, 384, 80, 1, 2),
    (61, 333, 96, 2, 1), (61, 333, 88, 2, 1), (17, 1024, 160, 2, 2), (29, 1024, 224, 1, 1)])
def test_key_groups_go_by_the_columns_multiplied(capi, heads, n, d, fwd, dq):
    """Odd numbers of heads at the column counts between the table's rows."""
    info = capi.launch_info(1, heads, n, n, d)
    assert (info["fwd"]["key_groups"], info["dq"]["key_groups"]) == (fwd, dq)


@pytest.mark.parametrize("heads,n,d,form", [
    (4, 16384, 48, "paired"), (4096, 640, 48, "paired"), (2048, 1024, 48, "paired"), (2048, 1025, 48, "direct"),
    (80, 3000, 48, "paired"), (80, 3000, 40, "paired"), (48, 4096, 48, "direct"), (32, 8192, 40, "direct"),
    (256, 1024, 64, "paired"), (80, 3000, 64, "direct"), (80, 3000, 56, "direct"), (2048, 640, 64, "direct"),
    (80, 3000, 32, "direct")])
def test_paired_dkdv_kernel_only_where_it_measured_faster(capi, heads, n, d, form):
    """The dK/dV kernel on both sides of the lines of the rows of 64 columns, whose 48-column form has its own."""
    assert capi.launch_info(1, heads, n, n, d)["dkdv"]["form"] == form


def test_traffic_stamp_ignores_comments_and_follows_code(tmp_path, monkeypatch):
    """bench.py drops the measured HBM traffic when the kernel sources have changed since the
    counter run.  The stamp it compares must not move when comments or layout change (nobody should
    have to re-stamp a summary by hand) and must move when code does."""
    import importlib

    bench = importlib.import_module("bench")
    src = tmp_path / "csrc"
    src.mkdir()
    (src / "k.hpp").write_text('// a comment\nint f(int x) { return x + 1; }  /* tail */\nconst char *s = "// not a comment";\n')
    (src / "Makefile").write_text("all:\n\ttrue\n")
    monkeypatch.setattr(bench, "KERNEL_SOURCES", src)
    base = bench.kernel_sources_hash()
    (src / "k.hpp").write_text('// another comment, more of it\n\nint f(int x)\n{\n  return x + 1;\n}\nconst char *s = "// not a comment";\n')
    assert bench.kernel_sources_hash() == base
    (src / "k.hpp").write_text('int f(int x) { return x + 2; }\nconst char *s = "// not a comment";\n')
    assert bench.kernel_sources_hash() != base
    (src / "k.hpp").write_text('int f(int x) { return x + 1; }\nconst char *s = "// not a comment!";\n')
    assert bench.kernel_sources_hash() != base
    # The committed summary carries the stamp of the committed sources.
    monkeypatch.undo()
    rows, source = bench._measured_traffic("C3")
    assert rows.get("fwd") and rows.get("bwd_dkdv") and rows.get("fwd_forward_only"), source
