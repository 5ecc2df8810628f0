"""The entry points as native calls (csrc/host_calls.cpp): ``_fast.fp8_gemm(a, b, a_s, b_s)`` and so on return the result of
the Python function of that name, or None without having done anything when the call is not a plain one; the Python function
then takes its own path.  The module is loaded at the first use.  It is built for one torch version, unlike the C library
behind both paths: without it (not built, or built for another torch) every call takes the Python path, after one warning."""
import importlib.util
import os
import warnings

from . import _lib
from ._build import HOST_PATH

# the library's entry points in the order of the Abi struct in csrc/host_calls.cpp
_ABI = ('dlb_last_error', 'dlb_workspace_lock', 'dlb_workspace_unlock', 'dlb_fp8_gemm', 'dlb_fp8_gemm_grouped_contiguous', 'dlb_fp8_gemm_grouped_contiguous_same_rows',
        'dlb_fp8_gemm_grouped_contiguous_gather_silu_quant', 'dlb_fp8_gemm_grouped_masked',
        'dlb_expert_gate_up_masked', 'dlb_fp8_gemm_grouped_ragged', 'dlb_expert_gate_up_ragged', 'dlb_expert_plan', 'dlb_fp8_quant_group',
        'dlb_silu_mul_quant_masked', 'dlb_ep_scatter_workspace_bytes', 'dlb_ep_scatter_rows_host', 'dlb_ep_gather')


_FUNCTIONS = ('fp8_gemm', 'quant', 'grouped_contiguous', 'grouped_masked', 'low_latency_experts', 'ep_gather', 'fused_moe_v3')


def _declined(*args):
    return None


def _load():
    import ctypes
    lib = _lib.load()
    try:
        if not os.path.exists(HOST_PATH):
            raise ImportError('it has not been built')
        spec = importlib.util.spec_from_file_location('dlblas_amd._host', HOST_PATH)
        host = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(host)
        host.init([ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in _ABI], _lib.workspace)
    except (ImportError, ValueError) as exc:
        warnings.warn(f'cannot use {HOST_PATH} ({exc}): calls cost more host time; run `python -m dlblas_amd._build`', RuntimeWarning)
        return None
    return host


def __getattr__(name):
    if name not in _FUNCTIONS:
        raise AttributeError(name)
    try:
        host = _load()
    except ImportError:  # no library: the Python path says so as soon as it needs it
        return _declined
    for fn in _FUNCTIONS:
        globals()[fn] = getattr(host, fn) if host is not None else _declined
    return globals()[name]
