"""The weight-streaming kernel of the masked layout (csrc/fp8_gemm_stream.h) at the sizes where it can go wrong: rows
around the edges of its tiles and fragments, several row tiles per expert, more experts than a wave has lanes, ragged N,
K as short as its ring and around the chunks of its scale table, both scale layouts and both output types.  It adds a K
block's products in the order of the ring kernels, so every shape has to give their bits."""
import pytest
import torch

import helpers
from oracle import fp8_block_gemm as orc

pytestmark = pytest.mark.gpu

SHAPES = ['32x256', '64x256', '64x128', '128x256', '64x64']


@pytest.fixture(scope='module')
def dev():
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    return torch.device('cuda:0')


def _inputs(masked, M_max, N, K, seed, dev):
    G = len(masked)
    g = helpers.gen(seed)
    a_q, a_s = orc.quant_act_1x128(torch.randn(G, M_max, K, generator=g).to(torch.bfloat16))
    ws = [orc.quant_weight_128x128((torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16)) for _ in range(min(G, 5))]
    w_q, w_s = (torch.stack([ws[e % len(ws)][i] for e in range(G)]) for i in (0, 1))
    bits = a_q.view(torch.uint8).clone()
    for e, m in enumerate(masked):  # rows past the valid ones: NaN codes and scales
        bits[e, m:] = 0x7F
        a_s[e, m:] = float('nan')
    a_q = bits.view(torch.float8_e4m3fn)
    return a_q.to(dev), a_s.to(dev), w_q.to(dev), w_s.to(dev), torch.tensor(masked, dtype=torch.int32, device=dev)


@pytest.mark.parametrize('masked,M_max,N,K,out_dtype,col_major', [
    ([1, 31, 32, 33, 0, 64], 64, 256, 1280, torch.bfloat16, False),     # 10 K blocks: as short as the deepest ring allows + 2
    ([65, 127, 128, 129, 3], 136, 520, 2176, torch.bfloat16, True),     # 17 blocks: two chunks of the table; ragged N
    ([5, 200, 0, 17], 200, 130, 1152, torch.float32, False),            # N no multiple of 8: element stores
    ([i % 4 for i in range(70)], 8, 128, 1024, torch.float32, True),    # a second window of 64 experts
    ([0, 0, 0], 32, 256, 1024, torch.bfloat16, False),                  # nothing to do
    ([40, 100], 100, 384, 256, torch.bfloat16, False),                  # 2 K blocks: only the three-stage rings
])
def test_masked_equals_the_ring_kernels(dev, masked, M_max, N, K, out_dtype, col_major):
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_masked
    a_q, a_s, w_q, w_s, mm = _inputs(masked, M_max, N, K, 40 + N + K, dev)
    if col_major:
        a_s = a_s.transpose(1, 2).contiguous().transpose(1, 2)
    outs = []
    for knob in [1] + [2 + i for i in range(len(SHAPES))]:
        print(f'case stream masked={masked[:6]} M_max={M_max} N={N} K={K} {out_dtype} shape={"ring" if knob == 1 else SHAPES[knob - 2]}', flush=True)
        out = torch.full((len(masked), M_max, N), -555.0, dtype=out_dtype, device=dev)
        _lib.tune('stream', knob)
        m_grouped_fp8_gemm_nt_masked((a_q, a_s), (w_q, w_s), out, mm, 0)
        torch.cuda.synchronize()
        _lib.tune('stream', 0)
        outs.append(out)
    for shape, out in zip(SHAPES, outs[1:]):
        assert torch.equal(out, outs[0]), shape
    ref = orc.grouped_masked_ref(a_q.cpu(), a_s.cpu(), w_q.cpu(), w_s.cpu(), torch.full((len(masked), M_max, N), -555.0), mm.cpu())
    valid = torch.arange(M_max)[None, :] < mm.cpu()[:, None]
    assert (outs[1].cpu()[~valid] == -555.0).all()
    if valid.any():
        helpers.tolerance_check(outs[1].cpu()[valid], ref[valid], f'stream {N}x{K}')


@pytest.mark.parametrize('masked,M_max,inter,K', [
    ([1, 32, 33, 0, 128, 64], 128, 256, 512),
    ([130, 5], 160, 128, 2304),
    ([i % 3 for i in range(66)], 4, 128, 384),
])
def test_masked_activation_equals_the_ring_kernel(dev, masked, M_max, inter, K):
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import fp8_gemm_grouped_masked_silu_quant
    a_q, a_s, w_q, w_s, mm = _inputs(masked, M_max, 2 * inter, K, 60 + inter + K, dev)
    G = len(masked)
    outs = []
    for knob in (1, 2, 3, 5):  # the ring kernel and the shapes with 256 weight rows
        print(f'case stream act masked={masked[:6]} M_max={M_max} I={inter} K={K} knob={knob}', flush=True)
        q = torch.full((G, M_max, inter), 0x5a, dtype=torch.uint8, device=dev)
        s = torch.full((G, M_max, inter // 128), -7.0, device=dev)
        _lib.tune('stream', knob)
        assert fp8_gemm_grouped_masked_silu_quant(a_q, a_s, w_q, w_s, q.view(torch.float8_e4m3fn), s, mm)
        torch.cuda.synchronize()
        _lib.tune('stream', 0)
        outs.append((q, s))
    for q, s in outs[1:]:
        assert torch.equal(q, outs[0][0]) and torch.equal(s, outs[0][1])
