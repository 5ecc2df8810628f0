"""The dense kernel whose waves split K (csrc/fp8_gemm_wavek.h): every tile shape at the edges of its tiles, with fewer K
blocks than waves, a ragged last K block, ragged N, both output types and strided scales, against the exact oracle; and the
library's choice of it."""
import ctypes

import pytest
import torch

import helpers
from oracle import fp8_block_gemm as orc

pytestmark = pytest.mark.gpu

N_SHAPES = 7


@pytest.fixture(scope='module')
def dev():
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    return torch.device('cuda:0')


def _operands(M, N, K, seed):
    g = helpers.gen(seed)
    whole = -(-K // 128) * 128
    a, a_s = orc.quant_act_1x128(torch.randn(M, whole, generator=g).to(torch.bfloat16))
    b, b_s = orc.quant_weight_128x128((torch.randn(N, whole, generator=g) * 0.05).to(torch.bfloat16))
    return a[:, :K].contiguous(), b[:, :K].contiguous(), a_s, b_s


@pytest.mark.parametrize('M,N,K', [
    (1, 32, 128),        # one block: every wave but one has nothing to do
    (33, 100, 384),      # rows one past a fragment, N no multiple of 8
    (64, 136, 1040),     # ragged K: one chunk in the last block
    (65, 72, 2032),      # ragged K: one chunk missing
    (130, 264, 1152),    # one block more than eight waves take in a round
    (97, 128, 16),       # K of one chunk
])
@pytest.mark.parametrize('out_dtype', [torch.bfloat16, torch.float32])
def test_every_shape_matches_the_oracle(dev, M, N, K, out_dtype):
    from dlblas_amd import _lib
    lib = _lib.load()
    a, b, a_s, b_s = _operands(M, N, K, M + N + K)
    ref = orc.dequant_ref(a, a_s, b, b_s)
    a, b, b_s = a.to(dev), b.to(dev), b_s.to(dev)
    by_row, by_block = a_s.to(dev), a_s.to(dev).t().contiguous().t()  # scales of a row / of a K block contiguous
    ws = _lib.workspace(dev, torch.cuda.current_stream().cuda_stream)
    vp = ctypes.c_void_p
    for shape in range(N_SHAPES):
        outs = []
        for s in (by_row, by_block):
            print(f'case wave_k {M}x{N}x{K} {out_dtype} shape {shape} strides {s.stride()}', flush=True)
            out = torch.full((M + 1, N), -555.0, dtype=out_dtype, device=dev)  # a guard row behind the result
            _lib.tune('wave_k', 2 + shape)
            _lib.check(lib.dlb_fp8_gemm(vp(a.data_ptr()), vp(b.data_ptr()), vp(s.data_ptr()), vp(b_s.data_ptr()), vp(out.data_ptr()), M, N, K,
                                        s.stride(0), s.stride(1), _lib.out_code(out_dtype), vp(ws.data_ptr()), ws.numel(),
                                        vp(torch.cuda.current_stream().cuda_stream)))
            torch.cuda.synchronize()
            _lib.tune('wave_k', 0)
            outs.append(out)
        assert torch.equal(outs[0], outs[1]) and (outs[0][M] == -555.0).all()
        helpers.tolerance_check(outs[0][:M], ref, f'wave_k shape {shape} {M}x{N}x{K}')


@pytest.mark.parametrize('M,N,K', [(100, 2112, 7168), (300, 1000, 1040), (500, 4096, 7168)])
def test_library_choice_full_size(dev, M, N, K):
    """Sizes the library gives to this kernel: sampled rows against the oracle; two calls agree bit for bit."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm import fp8_gemm
    print(f'case wave_k choice {M}x{N}x{K}', flush=True)
    plan = _lib.plan_wave_k(M, N, K)
    assert plan is not None and _lib.plan_wave_k(4096, 7168, 18432) is None and _lib.plan_wave_k(16, 7168, 2048) is None
    a, b, a_s, b_s = _operands(M, N, K, 3)
    prev = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        out = fp8_gemm(a.to(dev), b.to(dev), a_s.to(dev), b_s.to(dev))
        again = fp8_gemm(a.to(dev), b.to(dev), a_s.to(dev), b_s.to(dev))
    finally:
        torch.set_default_dtype(prev)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    rows = [0, 31, 32, M // 2, M - 1]
    helpers.tolerance_check(out[rows], orc.dequant_ref(a[rows], a_s[rows], b, b_s), f'wave_k {M}x{N}x{K}')


def test_scales_further_apart_than_32_bit_offsets(dev):
    """1023 K blocks whose scales lie up to 4.5 GB behind a tile's first one: beyond what the scale table's fetch can address,
    so the launch goes to a kernel with 64-bit addressing."""
    from dlblas_amd import _lib
    lib = _lib.load()
    M, N, K, sm, sk = 33, 32, 1023 * 128, (1 << 21) - 1, (1 << 20) - 1
    print(f'case wave_k far scales {M}x{N}x{K}', flush=True)
    a, b, a_s, b_s = _operands(M, N, K, 8)
    ref = orc.dequant_ref(a, a_s, b, b_s)
    far = torch.zeros((M - 1) * sm + (K // 128 - 1) * sk + 1, device=dev).as_strided((M, K // 128), (sm, sk))
    far.copy_(a_s)
    a, b, b_s = a.to(dev), b.to(dev), b_s.to(dev)
    ws = _lib.workspace(dev, torch.cuda.current_stream().cuda_stream)
    vp = ctypes.c_void_p
    out = torch.empty(M, N, device=dev)
    _lib.check(lib.dlb_fp8_gemm(vp(a.data_ptr()), vp(b.data_ptr()), vp(far.data_ptr()), vp(b_s.data_ptr()), vp(out.data_ptr()), M, N, K, sm, sk,
                                _lib.OUT_F32, vp(ws.data_ptr()), ws.numel(), vp(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    helpers.tolerance_check(out, ref, f'wave_k far scales {M}x{N}x{K}')
