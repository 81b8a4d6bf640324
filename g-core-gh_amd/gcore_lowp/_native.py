"""The native front end of the calls made most often (csrc/host/native.cpp), loaded on first use.

`fast.NAME(...)` returns the result, or None when the call is not the plain one it takes (see there): the wrapper then goes its
own way.  An eager quantise-and-multiply of one row took 26 us of host time through the interpreter and ctypes."""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import os

from . import _abi as A

PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_lib", "_lowp_native.so")
_BOUND = ("lp_quant_fp8_block", "lp_dequant_fp8_block", "lp_dequant_fp4_block", "lp_fp4_to_fp8_amax", "lp_fp4_to_fp8_rebase",
          "lp_gemm_fp8_block", "lp_gemm_workspace_bytes", "lp_host_flag")


def _load():
    lib = A.lib()
    if not os.path.exists(PATH):
        raise A.LowpError(f"{PATH} is missing: build it with `python g-core-gh_amd/build.py`")
    loader = importlib.machinery.ExtensionFileLoader("_lowp_native", PATH)
    mod = importlib.util.module_from_spec(importlib.util.spec_from_file_location("_lowp_native", PATH, loader=loader))
    loader.exec_module(mod)
    mod.bind(*(ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _BOUND))
    return mod


class _Fast:
    def __getattr__(self, name):                    # the first use of any entry
        mod = _load()
        for n in ("quant_fp8", "dequant", "fp4_to_fp8", "gemm"):
            setattr(self, n, getattr(mod, n))
        return getattr(mod, name)


fast = _Fast()
