"""The native front end of the calls made most often (csrc/host/native.cpp), loaded on first use.

`fast.NAME(...)` returns the result, or None when the call is not the plain one it takes (see there): the wrapper then goes its
own way.  An eager quantise-and-multiply of one row took 26 us of host time through the interpreter and ctypes.

The extension is compiled against one torch and one Python.  Where it is missing, does not load or was built for others, a warning
says so once and every call goes the wrapper's way: the same kernels through the C ABI alone."""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import os
import sysconfig
import warnings

import torch

from . import _abi as A

PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_lib", "_lowp_native.so")
_BOUND = ("lp_quant_fp8_block", "lp_dequant_fp8_block", "lp_dequant_fp4_block", "lp_fp4_to_fp8_amax", "lp_fp4_to_fp8_rebase",
          "lp_gemm_fp8_block", "lp_gemm_block_workspace_bytes", "lp_host_flag", "lp_host_table", "lp_quant_fp8_row_colwise_t",
          "lp_gemm_fp8_grouped", "lp_gemm_fp8_grouped_nn", "lp_gemm_fp8_rowscale_grouped", "lp_zero_slots", "lp_gemm_fp8_grouped_rows")
_ENTRIES = ("quant_fp8", "dequant", "fp4_to_fp8", "gemm", "grouped_forward", "grouped_backward")


def built_for() -> str:
    """What an extension has to be built for to be used here (g-core-gh_amd/build.py says it to the compiler)."""
    return f"torch {torch.__version__} {torch.version.git_version} {sysconfig.get_config_var('SOABI')}"


def _load():
    """The extension, bound to the library; ImportError if there is none for this torch and Python."""
    lib = A.lib()
    if not os.path.exists(PATH):
        raise ImportError(f"{PATH} is missing")
    loader = importlib.machinery.ExtensionFileLoader("_lowp_native", PATH)
    mod = importlib.util.module_from_spec(importlib.util.spec_from_file_location("_lowp_native", PATH, loader=loader))
    loader.exec_module(mod)
    if getattr(mod, "built_for", None) != built_for():
        raise ImportError(f"{PATH} was built for {getattr(mod, 'built_for', 'another torch')}, this is {built_for()}")
    mod.bind(*(ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _BOUND))
    return mod


class _Fast:
    def __getattr__(self, name):                    # the first use of any entry
        if name not in _ENTRIES:
            raise AttributeError(name)
        try:
            mod = _load()
        except ImportError as e:
            warnings.warn(f"{e}: calls take about 10 us more of host time; build it with `python g-core-gh_amd/build.py`", RuntimeWarning,
                          stacklevel=3)
            for n in _ENTRIES:
                setattr(self, n, lambda *args: None)
            return getattr(self, name)
        for n in _ENTRIES:
            setattr(self, n, getattr(mod, n))
        return getattr(mod, name)


fast = _Fast()
