"""ctypes binding of libfa2_gfx950.so (declarations: include/fa2_gfx950.h).

The binding passes raw device pointers, sizes, element strides and the current HIP stream; it
holds no torch types in any signature.  There is no CPU or PyTorch fallback: if the library is
missing or reports an error, the caller gets an exception.
"""

from __future__ import annotations

import ctypes
import os
import pathlib
import threading

# The in-tree build; FA2_GFX950_LIBRARY names another build of the same ABI (e.g. one under test).
LIBRARY_PATH = pathlib.Path(os.environ.get("FA2_GFX950_LIBRARY") or
                            pathlib.Path(__file__).resolve().parent / "csrc" / "libfa2_gfx950.so")
ABI_VERSION = 9

FA2_DTYPE_F16 = 0
FA2_DTYPE_BF16 = 1
FA2_CONFIG_AUTO = -1
FA2_MAX_HEADDIM = 256
FA2_NOALLOC_MAX_ROWS = 4 << 20

_i, _i64, _f, _p = ctypes.c_int, ctypes.c_int64, ctypes.c_float, ctypes.c_void_p


class ConfigInfo(ctypes.Structure):
    """Mirror of ``fa2_config_info``: one row of the gfx950 tile/wave table."""

    _fields_ = [(name, ctypes.c_int) for name in (
        "id", "headdim_padded",
        "fwd_block_q", "fwd_block_kv", "fwd_waves",
        "bwd_block_q", "bwd_block_kv", "bwd_waves",
        "dq_block_q", "dq_block_kv", "dq_waves",
        "lds_direct", "fwd_wg_per_cu", "dq_wg_per_cu", "dkdv_wg_per_cu",
        "lds_stages", "dkdv_passes", "head_group", "dq_atomic", "fwd_exp_folded")]

    def as_dict(self) -> dict:
        return {name: getattr(self, name) for name, _ in self._fields_}


class LaunchPart(ctypes.Structure):
    """Mirror of ``fa2_launch_part``: form, tile and grid of one kernel of a call."""

    _fields_ = [*((name, _i) for name in ("form", "block_rows", "key_groups", "wg_per_cu", "resident")),
                ("workgroups", _i64)]

    def as_dict(self) -> dict:
        return {**{name: getattr(self, name) for name, *_ in self._fields_}, "form": FORMS[self.form]}


class LaunchInfo(ctypes.Structure):
    """Mirror of ``fa2_launch_info``."""

    _fields_ = [("config_id", _i), ("fwd", LaunchPart), ("dq", LaunchPart), ("dkdv", LaunchPart)]


class Tensor(ctypes.Structure):
    """Mirror of ``fa2_tensor``: device pointer and the batch, head and sequence strides in elements."""

    _fields_ = [("ptr", _p), ("stride_batch", _i64), ("stride_head", _i64), ("stride_seq", _i64)]


class FwdArgs(ctypes.Structure):
    """Mirror of ``fa2_fwd_args``."""

    _fields_ = [("q", Tensor), ("k", Tensor), ("v", Tensor), ("o", Tensor), ("lse", _p),
                ("batch", _i), ("nheads", _i), ("seqlen_q", _i), ("seqlen_k", _i), ("headdim", _i),
                ("seqlen_q_rounded", _i), ("softmax_scale", _f), ("dtype", _i), ("config_id", _i)]


class Cast(ctypes.Structure):
    """Mirror of ``fa2_cast``."""

    _fields_ = [("src", _p), ("dst", _p), ("n", _i64)]


class BwdArgs(ctypes.Structure):
    """Mirror of ``fa2_bwd_args``."""

    _fields_ = [("q", Tensor), ("k", Tensor), ("v", Tensor), ("o", Tensor), ("d_o", Tensor),
                ("dq", Tensor), ("dk", Tensor), ("dv", Tensor), ("lse", _p), ("delta", _p),
                ("workspace", _p),
                ("batch", _i), ("nheads", _i), ("seqlen_q", _i), ("seqlen_k", _i), ("headdim", _i),
                ("seqlen_q_rounded", _i), ("softmax_scale", _f), ("dtype", _i), ("deterministic", _i),
                ("config_id", _i)]


# Every symbol include/fa2_gfx950.h declares, with its ctypes signature.
SIGNATURES = {
    "fa2_abi_version": (_i, []),
    "fa2_last_error_string": (ctypes.c_char_p, []),
    "fa2_status_string": (ctypes.c_char_p, [_i]),
    "fa2_config_count": (_i, []),
    "fa2_config_get": (_i, [_i, ctypes.POINTER(ConfigInfo)]),
    "fa2_pick_config": (_i, [_i, _i, _i, _i, _i]),
    "fa2_pick_config_forward_only": (_i, [_i, _i, _i, _i]),
    "fa2_fwd": (_i, [_p] * 5 + [_i] * 6 + [_i64] * 12 + [_f, _i, _i, _p]),
    "fa2_bwd_preprocess": (_i, [_p] * 3 + [_i] * 5 + [_i64] * 6 + [_i, _p]),
    "fa2_bwd_workspace_bytes": (ctypes.c_size_t, [_i] * 7),
    "fa2_bwd": (_i, [_p] * 10 + [_i] * 6 + [_i64] * 21 + [_f, _i, _i, _i, _p]),
    "fa2_bwd_fused": (_i, [_p] * 11 + [_i] * 6 + [_i64] * 24 + [_f, _i, _i, _i, _p]),
    "fa2_bwd_fused_noalloc": (_i, [_p] * 9 + [_i] * 6 + [_i64] * 24 + [_f, _i, _i, _i, _p]),
    "fa2_launch_info_get": (_i, [_i] * 6 + [ctypes.POINTER(LaunchInfo)]),
    "fa2_joint_info_get": (_i, [_i] * 6 + [ctypes.POINTER(LaunchPart)]),
    "fa2_fwd_packed": (_i, [ctypes.POINTER(FwdArgs), _p]),
    "fa2_fwd_packed_f32_out": (_i, [ctypes.POINTER(FwdArgs), _p, _p]),
    "fa2_cast_f32_to_f16": (_i, [ctypes.POINTER(Cast), _i, _p]),
    "fa2_bwd_packed": (_i, [ctypes.POINTER(BwdArgs), _p]),
    "fa2_bwd_packed_f32_grads": (_i, [ctypes.POINTER(BwdArgs), _p]),
}

_lib = None
_lock = threading.Lock()


def load() -> ctypes.CDLL:
    """Load the shared library once (thread-safe) and type every entry point."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is None:
            if not LIBRARY_PATH.exists():
                raise RuntimeError(
                    f"{LIBRARY_PATH} is missing: the HIP kernels are not built. "
                    "Build them with `python flash-attention-triton_amd/build.py` "
                    "(hipcc --offload-arch=gfx950); there is no fallback path."
                )
            lib = ctypes.CDLL(str(LIBRARY_PATH))
            lib.fa2_abi_version.restype = _i
            got = lib.fa2_abi_version()  # before the other symbols: a library of another version may lack some
            if got != ABI_VERSION:
                raise RuntimeError(f"libfa2_gfx950.so has ABI version {got}, binding expects {ABI_VERSION}")
            for name, (restype, argtypes) in SIGNATURES.items():
                fn = getattr(lib, name)
                fn.restype = restype
                fn.argtypes = argtypes
            _lib = lib
    return _lib


def check(status: int, what: str) -> None:
    """Turn a non-zero fa2_status into RuntimeError carrying the library's message."""
    if status != 0:
        lib = load()
        name = lib.fa2_status_string(status).decode()
        detail = lib.fa2_last_error_string().decode()
        raise RuntimeError(f"{what} failed: {name}: {detail}")


def config_table() -> list[dict]:
    lib = load()
    rows = []
    for i in range(lib.fa2_config_count()):
        info = ConfigInfo()
        check(lib.fa2_config_get(i, ctypes.byref(info)), "fa2_config_get")
        rows.append(info.as_dict())
    return rows


FORMS = ("generic", "direct", "paired", "mixed", "joint")


def launch_info(batch: int, nheads: int, seqlen_q: int, seqlen_k: int, headdim: int,
                config_id: int = FA2_CONFIG_AUTO) -> dict:
    """What a forward and a backward on contiguous tensors of these sizes launch (fa2_launch_info_get)."""
    info = LaunchInfo()
    check(load().fa2_launch_info_get(batch, nheads, seqlen_q, seqlen_k, headdim, config_id, ctypes.byref(info)),
          "fa2_launch_info_get")
    out = {"config_id": info.config_id}
    for part in ("fwd", "dq", "dkdv"):
        out[part] = getattr(info, part).as_dict()
    return out


def joint_info(batch: int, nheads: int, seqlen_q: int, seqlen_k: int, headdim: int,
               config_id: int = FA2_CONFIG_AUTO) -> dict | None:
    """The grid in which a backward of these sizes forms dq, dk and dv, None where two launches do (fa2_joint_info_get)."""
    part = LaunchPart()
    check(load().fa2_joint_info_get(batch, nheads, seqlen_q, seqlen_k, headdim, config_id, ctypes.byref(part)),
          "fa2_joint_info_get")
    return part.as_dict() if part.workgroups > 0 else None
