"""Loading of the native entry points (dlblas_amd/_fast.py): what happens without the module or without the library.  No GPU."""
import warnings

import pytest

from dlblas_amd import _fast, _lib


@pytest.fixture
def fresh(monkeypatch):
    """_fast as before its first use; restored afterwards."""
    for name in _fast._FUNCTIONS:
        monkeypatch.delitem(_fast.__dict__, name, raising=False)
    yield monkeypatch
    for name in _fast._FUNCTIONS:
        _fast.__dict__.pop(name, None)


@pytest.mark.parametrize('content', [None, b'not a library'])
def test_without_the_module_every_call_is_declined(fresh, tmp_path, content):
    path = tmp_path / '_host.so'
    if content is not None:
        path.write_bytes(content)
    fresh.setattr(_fast, 'HOST_PATH', str(path))
    with pytest.warns(RuntimeWarning, match='_host.so'):
        assert _fast.fp8_gemm(1, 2, 3, 4) is None
    with warnings.catch_warnings():
        warnings.simplefilter('error')  # one warning, not one a call
        for name in _fast._FUNCTIONS:
            assert getattr(_fast, name)() is None


def test_without_the_library_the_python_path_reports_it(fresh, tmp_path):
    import torch

    from dlblas_amd.kernels.fp8 import per_token_group_quant_fp8
    fresh.setattr(_lib, '_lib', None)
    fresh.setenv('DLBLAS_AMD_LIB', str(tmp_path / 'missing.so'))
    assert _fast.quant(torch.zeros(2, 128), 128, 1e-10, False) is None
    with pytest.raises(NotImplementedError):  # the op itself: no kernel for CPU tensors
        per_token_group_quant_fp8(torch.zeros(2, 128, dtype=torch.bfloat16), 128)
    with pytest.raises(ImportError, match='has not been built'):
        _lib.load()


def test_the_module_is_used_when_it_is_there(fresh):
    with warnings.catch_warnings():
        warnings.simplefilter('error')
        assert _fast.fp8_gemm is not _fast._declined
        assert _fast.fp8_gemm(1, 2, 3, 4) is None  # not tensors: left to the Python path


@pytest.mark.parametrize('form', [_lib.ON_ROW_RANGES, _lib.ON_WHOLE_BLOCKS])
def test_scales_between_the_expert_gemms_are_float32(form):
    """The kernels write 32 bits per scale, whatever the default dtype (it chooses the type fp8_gemm returns)."""
    import importlib

    import torch
    moe = importlib.import_module('dlblas_amd.kernels.fused_moe_v3')
    prev = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        s = moe._scales(256, 16, form, 'cpu')
    finally:
        torch.set_default_dtype(prev)
    assert s.dtype == torch.float32 and tuple(s.shape) == (256, 16) and s.untyped_storage().nbytes() == 256 * 16 * 4
    assert s.stride() == ((16, 1) if form == _lib.ON_ROW_RANGES else (1, 256))


@pytest.mark.parametrize('wrong,error', [
    ({}, RuntimeError),  # nothing but the device
    ({'out_s': lambda t: t.bfloat16()}, TypeError),
    ({'b_s': lambda t: t.double()}, TypeError),
    ({'row_start': lambda t: t.long()}, TypeError),
    ({'b': lambda t: t.transpose(1, 2).contiguous().transpose(1, 2)}, AssertionError),
    ({'b_s': lambda t: t[:, :1]}, AssertionError),
    ({'a_s': lambda t: t[:, :1]}, ValueError),
    ({'out_s': lambda t: t[:-1]}, ValueError),
    ({'out': lambda t: t[:-1]}, ValueError),
    ({'a_row_index': lambda t: t[:-1]}, ValueError),
])
def test_row_range_gemms_check_what_goes_behind_a_pointer(wrong, error):
    import torch
    f8 = lambda *s: torch.zeros(*s, dtype=torch.uint8).view(torch.float8_e4m3fn)
    args = dict(a=f8(5, 256), b=f8(2, 512, 256), a_s=torch.ones(5, 2), b_s=torch.ones(2, 4, 2), out=f8(256, 256), out_s=torch.ones(2, 256).t(),
                row_start=torch.zeros(2, dtype=torch.int32), row_end=torch.zeros(2, dtype=torch.int32),
                a_row_index=torch.zeros(256, dtype=torch.int32))
    for name, change in wrong.items():
        args[name] = change(args[name])
    for call in (_lib.expert_gate_up_ragged, _lib.gemm_ragged_silu_quant):
        with pytest.raises(error):
            call(*(args[n] for n in ('a', 'b', 'a_s', 'b_s', 'out', 'out_s', 'row_start', 'row_end', 'a_row_index')), 64, 1e-10)
