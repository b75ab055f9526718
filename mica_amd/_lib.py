"""ctypes binding of libmica_amd.so, the C ABI declared in include/mica_amd.h, and the loader of the native
launch path over it (binding/native.cpp, _native.so).

The library is loaded after torch, so it binds to the HIP runtime torch already loaded (same soname)
and the stream handles torch hands out are valid in it.  A missing library is an error, never a
silent fallback: build it with ``python -m mica_amd.build``.  Without the launch path calls go through Python,
with a warning.
"""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import os
import threading
import warnings
from pathlib import Path

LIB_NAME = "libmica_amd.so"
ENV_DIR = "MICA_AMD_LIB_DIR"
# always the package's own (its functions' arguments are those the package's Python files pass), whatever ENV_DIR names
NATIVE_PATH = Path(__file__).resolve().parent / "_native.so"

# dtype codes (mica_amd.h)
BF16, FP16, FP32, INT8, INT32 = 0, 1, 2, 3, 4
ROUND_EVEN, ROUND_AWAY = 0, 1
EPI_SCALE, EPI_SILU_MUL = 0, 1

MISS_NAMES = {1: "shape", 2: "dtype", 3: "align", 4: "stride", 5: "i32_range", 6: "arg", 7: "device"}

_P = ctypes.c_void_p
_I = ctypes.c_int
_F = ctypes.c_float
_LL = ctypes.c_longlong

# name -> (restype, argtypes); the order of arguments is that of include/mica_amd.h
SIGNATURES = {
    "mica_version": (_I, []),
    "mica_status_name": (ctypes.c_char_p, [_I]),
    "mica_device_info": (_I, [_I, ctypes.POINTER(_I), ctypes.POINTER(_I), ctypes.POINTER(_I), ctypes.POINTER(_I)]),
    "mica_act_quant": (_I, [_P, _I, _I, _P, _P, _I, _P, _I, _I, _I, _P]),
    "mica_rmsnorm_quant": (_I, [_P, _I, _I, _P, _I, _P, _I, _F, _F, _P, _P, _I, _P, _P, _I, _P, _I, _I, _I, _I,
                                _P]),
    "mica_rmsnorm_quant_multi": (_I, [_P, _I, _I, _P, _I, _P, _I, _F, _F, _I, _P, _P, _P, _P, _P, _I, _P, _I, _I, _I,
                                      _I, _P]),
    "mica_mm_i8": (_I, [_P, _I, _P, _I, _P, _P, _P, _P, _I, _P, _I, _I, _I, _I, _I, _I, _P, _LL, _P]),
    "mica_mm_i8_workspace_bytes": (_LL, [_I]),
    "mica_mm_i8_few_rows_tile": (_I, [_I, _I, _I, _I, _I, ctypes.POINTER(_I)]),
    "mica_mm_i8_noalloc": (_I, [_P, _I, _P, _I, _P, _P, _P, _P, _I, _P, _I, _I, _I, _I, _I, _I, _P]),
    "mica_mm_i8_noalloc_scratch_bytes": (_LL, []),
    "mica_swiglu": (_I, [_P, _P, _P, _LL, _I, _P]),
    "mica_gather_logits": (_I, [_P, _I, _I, _P, _I, _P, _I, _F, _F, _P, _I, _I, _I, _P, _I, _I, _P, _P, _P, _P, _I,
                                _P]),
    "mica_rope_inplace": (_I, [_P, _LL, _I, _I, _P, _P, _I, _P, _I, _I, _P]),
    "mica_head_norm_rope": (_I, [_P, _LL, _I, _I, _I, _I, _I, _I, _P, _P, _F, _F, _I, _P, _P, _I, _P, _I, _P]),
    "mica_gate_quant": (_I, [_P, _LL, _P, _LL, _P, _LL, _P, _P, _LL, _I, _I, _I, _P]),
    "mica_attention_fwd": (_I, [_P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _I, _I,
                                _I, _I, _I, _I, _F, _I, _P, _LL, _P]),
    "mica_attention_workspace_bytes": (_LL, [_I, _I, _I]),
    "mica_attention_fwd_split": (_I, [_P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _I,
                                      _I, _I, _I, _I, _I, _F, _I, _I, _P, _LL, _P]),
    "mica_attention_split_workspace_bytes": (_LL, [_I, _I, _I, _I, _I, _I]),
    "mica_attention_fwd_kvlen": (_I, [_P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _I,
                                      _I, _I, _I, _I, _I, _F, _I, _I, _P, _P, _LL, _P]),
    "mica_attention_fwd_prefix": (_I, [_P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _P, _LL, _LL, _P, _LL,
                                       _LL, _I, _P, _LL, _LL, _LL, _I, _I, _I, _I, _I, _I, _F, _I, _I, _P, _P, _LL,
                                       _P]),
    "mica_attention_prefix_workspace_bytes": (_LL, [_I, _I, _I, _I, _I, _I, _I]),
    "mica_attention_pipelined": (_I, [_I, _I, _I, _I, _I]),
    "mica_attention_fwd_rope": (_I, [_P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _P, _LL, _LL, _LL, _P, _LL, _LL, _P, _LL,
                                     _LL, _I, _P, _LL, _LL, _LL, _I, _I, _I, _I, _I, _I, _F, _I, _I, _P, _P, _F, _F,
                                     _I, _P, _P, _I, _P, _P, _LL, _P]),
    "mica_causal_conv1d": (_I, [_P, _LL, _I, _P, _P, _I, _I, _P, _P, _P, _LL, _I, _I, _I, _I, _I, _I, _F, _P]),
    "mica_gdn_chunk": (_I, [_P, _LL, _I, _P, _LL, _I, _P, _LL, _I, _P, _P, _I, _P, _P, _P, _F, _I, _I, _I, _I, _P,
                            _LL, _P]),
    "mica_gdn_chunk_gate": (_I, [_P, _LL, _I, _P, _LL, _I, _P, _LL, _I, _P, _I, _P, _I, _P, _P, _P, _P, _P, _F, _I, _I, _I,
                                 _I, _P, _LL, _P]),
    "mica_gdn_workspace_bytes": (_LL, [_I, _I, _I]),
    "mica_gated_rmsnorm_quant": (_I, [_P, _I, _P, _I, _P, _F, _P, _I, _P, _I, _P, _I, _I, _P]),
    "mica_gdn_gate": (_I, [_P, _I, _P, _I, _P, _P, _P, _P, _I, _I, _P]),
}

# functions of libmica_amd.so that the native launch path calls
NATIVE_FNS = ("mica_act_quant", "mica_mm_i8", "mica_rmsnorm_quant", "mica_rmsnorm_quant_multi",
              "mica_attention_prefix_workspace_bytes", "mica_attention_fwd", "mica_attention_fwd_prefix",
              "mica_causal_conv1d", "mica_gdn_chunk", "mica_gdn_chunk_gate", "mica_gdn_workspace_bytes",
              "mica_gdn_gate", "mica_gated_rmsnorm_quant")


class _NotLoaded:
    """Stands for the native launch path until load(), or where it does not load: every function declines the call."""

    def __getattr__(self, name):
        return lambda *args: None


# binding/native.cpp's functions: each launches a plain call and returns its result, or None for a call that the
# Python path has to serve or refuse, or the negative error of a failed launch (int)
FAST = _NotLoaded()

_LIB = None
_LOCK = threading.Lock()


def lib_path() -> Path:
    d = os.environ.get(ENV_DIR)
    return (Path(d) if d else Path(__file__).resolve().parent) / LIB_NAME


def _load_native(lib):
    """The launch path over `lib`, or its stand-in when the module is missing or does not load under this torch and
    Python: the Python path serves every call, so that is a warning about host time and no error."""
    try:
        loader = importlib.machinery.ExtensionFileLoader("mica_amd._native", str(NATIVE_PATH))
        mod = importlib.util.module_from_spec(importlib.util.spec_from_loader("mica_amd._native", loader))
        loader.exec_module(mod)
    except (ImportError, OSError) as exc:
        warnings.warn(f"mica_amd: no native launch path ({exc}); calls take 10 to 100 us more host time each. Rebuild "
                      "with `python -m mica_amd.build`", RuntimeWarning, stacklevel=3)
        return _NotLoaded()
    mod.bind({n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in NATIVE_FNS})
    return mod


def load():
    """Load (once) and return the ctypes library; raises RuntimeError if it is not built."""
    global _LIB, FAST
    if _LIB is not None:
        return _LIB
    with _LOCK:
        if _LIB is None:
            import torch  # noqa: F401  -- bind to torch's HIP runtime (see module docstring)

            path = lib_path()
            if not path.is_file():
                raise RuntimeError(f"{path} is not built; run `python -m mica_amd.build`")
            lib = ctypes.CDLL(str(path))
            for name, (res, args) in SIGNATURES.items():
                fn = getattr(lib, name)
                fn.restype, fn.argtypes = res, args
            FAST = _load_native(lib)
            _LIB = lib
    return _LIB


def status_name(rc: int) -> str:
    if rc > 0:
        return MISS_NAMES.get(rc, f"miss{rc}")
    return load().mica_status_name(rc).decode()


def check(rc: int, what: str) -> int:
    """Raise on a HIP error (rc < 0); return rc (0 = launched, > 0 = miss code)."""
    if rc < 0:
        raise RuntimeError(f"{what} failed: HIP error {-rc} {status_name(rc)}")
    return rc


def device_info(index: int = 0) -> dict:
    cu, clk, lds, arch = _I(), _I(), _I(), _I()
    check(load().mica_device_info(index, ctypes.byref(cu), ctypes.byref(clk), ctypes.byref(lds),
                                  ctypes.byref(arch)), "mica_device_info")
    return {"cu_count": cu.value, "clock_khz": clk.value, "lds_per_block": lds.value, "gfx_arch": arch.value}
