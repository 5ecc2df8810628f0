"""GPU parity of the HIP kernels (through the Python entry points -> C ABI) against the CPU oracle."""
import pytest
import torch

import helpers
from oracle import fp8_block_gemm as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def dev():
    import dlblas_amd  # noqa: F401
    from dlblas_amd import _lib
    _lib.load()
    return torch.device('cuda:0')


def _run_dense(dev, a_q, a_s, b_q, b_s, dtype=torch.bfloat16, variant=None):
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm import fp8_gemm
    prev = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        _lib.force_variant(variant)
        out = fp8_gemm(a_q.to(dev), b_q.to(dev), a_s.to(dev), b_s.to(dev))
        torch.cuda.synchronize()
    finally:
        _lib.force_variant(None)
        torch.set_default_dtype(prev)
    return out


def _run_dense_guarded(dev, a_q, a_s, b_q, b_s, dtype=torch.bfloat16, variant=None, first=0):
    """The result written from element `first` of a buffer on; the elements before and behind it have to stay as they were."""
    import ctypes

    from dlblas_amd import _lib
    (M, K), N, vp = a_q.shape, b_q.size(0), ctypes.c_void_p
    a, b, sa, sb = (t.to(dev) for t in (a_q, b_q, a_s, b_s))
    whole = torch.full((first + M * N + 64, ), -777.0, dtype=dtype, device=dev)
    stream = torch.cuda.current_stream().cuda_stream
    ws = _lib.workspace(dev, stream)
    try:
        _lib.force_variant(variant)
        rc = _lib.load().dlb_fp8_gemm(vp(a.data_ptr()), vp(b.data_ptr()), vp(sa.data_ptr()), vp(sb.data_ptr()),
                                      vp(whole.data_ptr() + first * whole.element_size()), M, N, K, sa.stride(0), sa.stride(1),
                                      _lib.OUT_F32 if dtype == torch.float32 else _lib.OUT_BF16, vp(ws.data_ptr()), ws.numel(), vp(stream))
        torch.cuda.synchronize()
    finally:
        _lib.force_variant(None)
    assert rc == 0, _lib.last_error()
    assert bool((whole[:first] == -777.0).all()) and bool((whole[first + M * N:] == -777.0).all()), f'{variant}: written beside the result'
    return whole[first:first + M * N].view(M, N)


DENSE_SHAPES = [
    (64, 512, 1024),      # the reference's CPU-runnable configuration
    (512, 512, 512),      # the shape of tests/kernels/test_fp8_gemm.py
    (1, 7168, 2048), (16, 7168, 2048), (64, 7168, 2048), (128, 7168, 2048),
    (1, 2112, 7168), (16, 2112, 7168), (64, 2112, 7168), (128, 2112, 7168),
    (16, 1000, 640), (1, 392, 896), (32, 520, 512),  # decode with 4 to 7 K blocks: 8 waves, some of them without a block
    (300, 2112, 1536),    # ragged M and N tiles
    (256, 7168, 2048), (384, 2112, 7168), (130, 7168, 16384),  # between decode and prefill: small tiles, K split over workgroups
    (129, 130, 384),      # N not a multiple of 4: scalar stores
    (33, 200, 400),       # K tail (400 = 3 * 128 + 16)
    (17, 64, 200),        # K not a multiple of 16: exact path
]


@pytest.mark.parametrize('M,N,K', DENSE_SHAPES)
def test_dense_bf16_matches_oracle(dev, M, N, K):
    print(f'case dense bf16 M={M} N={N} K={K}', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(M, N, K)
    ref = orc.dequant_ref(a_q, a_s, b_q, b_s)
    out = _run_dense(dev, a_q, a_s, b_q, b_s)
    assert out.dtype == torch.bfloat16 and tuple(out.shape) == (M, N)
    helpers.tolerance_check(out, ref, f'dense {M}x{N}x{K}')


@pytest.mark.parametrize('variant', ['tile128x128', 'tile64x128', 'tile128x64', 'skinny16', 'skinny32', 'skinny64', 'skinny128', 'exact', 'pipe256x256', 'pipe128x256w8', 'pipe256mix', 'pipe128x128', 'pipe128x64'])
@pytest.mark.parametrize('M,N,K', [(16, 512, 1024), (30, 200, 400), (200, 392, 2048)])
def test_every_variant(dev, variant, M, N, K):
    print(f'case variant={variant} M={M} N={N} K={K}', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(M, N, K, seed=7)
    ref = orc.dequant_ref(a_q, a_s, b_q, b_s)
    out = _run_dense(dev, a_q, a_s, b_q, b_s, variant=variant)
    helpers.tolerance_check(out, ref, f'{variant} {M}x{N}x{K}')


@pytest.mark.parametrize('out_dtype', [torch.bfloat16, torch.float32])
@pytest.mark.parametrize('variant,splitk', [('tile128x128', 2), ('tile128x64', 5), ('tile64x128', 32), (None, 0), ('pipe128x256w8', 3),
                                            ('pipe128x128', 4), ('pipe128x64', 2), ('pipe256x256', 7)])
@pytest.mark.parametrize('M,N,K', [(128, 2112, 7168), (200, 392, 2048), (129, 130, 1040), (70, 131, 4096)])
def test_split_k_two_pass(dev, M, N, K, variant, splitk, out_dtype):
    """K split over workgroups: fp32 partial matrices in the workspace, a second kernel adds them in index order.
    (None, 0) is the library's own choice among the kernels that split K over workgroups.  Two
    calls must agree bit for bit."""
    from dlblas_amd import _lib
    print(f'case split-K variant={variant} splitk={splitk} M={M} N={N} K={K} {out_dtype}', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(M, N, K, seed=11)
    ref = orc.dequant_ref(a_q, a_s, b_q, b_s)
    try:
        _lib.force_splitk(splitk)
        _lib.tune('wave_k', 1 if variant is None else 0)
        assert variant is not None or _lib.plan(0, M, N, K)[1] > 1
        out = _run_dense(dev, a_q, a_s, b_q, b_s, dtype=out_dtype, variant=variant)
        again = _run_dense(dev, a_q, a_s, b_q, b_s, dtype=out_dtype, variant=variant)
    finally:
        _lib.force_splitk(0)
        _lib.tune('wave_k', 0)
    assert out.dtype == out_dtype
    helpers.tolerance_check(out, ref, f'split-K {variant}/{splitk} {M}x{N}x{K}')
    assert torch.equal(out, again)


@pytest.mark.parametrize('out_dtype', [torch.bfloat16, torch.float32])
@pytest.mark.parametrize('variant,splitk', [('pipe128x64', 7), ('pipe128x64', 2), ('pipe128x128', 4), ('pipe128x128', 32), ('pipe128x256w8', 3),
                                            ('pipe256x256', 5)])
@pytest.mark.parametrize('M,N,K', [(128, 2112, 7168), (200, 392, 2048), (129, 130, 4096), (33, 64, 4096)])
def test_split_k_in_one_launch_equals_two_pass(dev, M, N, K, variant, splitk, out_dtype):
    """The K slices of a tile added by its own workgroups (arrival counter in the workspace head, bounded wait, slices
    summed in index order) give the bits of the two-pass path; so does the path in which nobody waits and the workgroup
    that completes a tile adds every share (spin limit 0).  Every call leaves the counter head all zero."""
    from dlblas_amd import _lib
    print(f'case one-launch split-K variant={variant} splitk={splitk} M={M} N={N} K={K} {out_dtype}', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(M, N, K, seed=13)
    ref = orc.dequant_ref(a_q, a_s, b_q, b_s)
    head = _lib.workspace(dev, torch.cuda.current_stream().cuda_stream)[:_lib.WS_COUNTER_BYTES]
    outs = []
    try:
        _lib.force_splitk(splitk)
        for mode, spin in ((2, 0), (1, 0), (1, 1), (1, 0)):
            _lib.tune('splitk_mode', mode)
            _lib.tune('spin_limit', spin)
            outs.append(_run_dense(dev, a_q, a_s, b_q, b_s, dtype=out_dtype, variant=variant))
            assert int(head.count_nonzero()) == 0, f'counter head not zero after mode {mode} spin {spin}'
    finally:
        _lib.force_splitk(0)
        _lib.tune('splitk_mode', 0)
        _lib.tune('spin_limit', 0)
    helpers.tolerance_check(outs[0], ref, f'one-launch split-K {variant}/{splitk} {M}x{N}x{K}')
    for o in outs[1:]:
        assert torch.equal(o, outs[0])


@pytest.mark.parametrize('variant,splitk', [('pipe128x64', 0), ('pipe128x64', 7), ('pipe128x128', 2), ('pipe128x128', 5)])
@pytest.mark.parametrize('M,N,K', [(128, 2112, 7168), (256, 520, 2048), (77, 200, 4096), (300, 392, 1024)])
def test_scale_table_equals_scales_per_stage(dev, M, N, K, variant, splitk):
    """Row-major activation scales fetched once per tile into the table in LDS (the default of the small ring kernels up
    to 32 K blocks per workgroup) against the same kernels fetching them stage by stage: the same values, the same bits.
    Column-major scales never take the table."""
    from dlblas_amd import _lib
    print(f'case scale table variant={variant} splitk={splitk} M={M} N={N} K={K}', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(M, N, K, seed=19)
    ref = orc.dequant_ref(a_q, a_s, b_q, b_s)
    try:
        _lib.force_splitk(splitk)
        with_table = _run_dense(dev, a_q, a_s, b_q, b_s, variant=variant)
        _lib.tune('scale_table', 2)
        per_stage = _run_dense(dev, a_q, a_s, b_q, b_s, variant=variant)
    finally:
        _lib.force_splitk(0)
        _lib.tune('scale_table', 0)
    helpers.tolerance_check(with_table, ref, f'scale table {variant}/{splitk} {M}x{N}x{K}')
    assert torch.equal(with_table, per_stage)


@pytest.mark.parametrize('layout,variant,rows,N,blocks', [
    ('dense', 'pipe256x256', 300, 520, 27), ('dense', 'pipe256x256', 257, 130, 28), ('dense', 'pipe256mix', 700, 1000, 1),
    ('dense', 'pipe256mix', 513, 1000, 5), ('dense', 'pipe128x256w8', 257, 300, 5), ('dense', 'pipe128x256w8', 129, 300, 16),
    ('contiguous', 'pipe128x128', 512, 392, 54), ('contiguous', 'pipe128x128', 384, 136, 55), ('contiguous', 'pipe128x256w8', 640, 520, 16),
    ('masked', 'pipe128x128', 200, 392, 3), ('masked', 'pipe256x256', 300, 392, 27), ('masked', 'pipe256x256', 260, 130, 28)])
def test_scale_table_of_every_ring_kernel(dev, layout, variant, rows, N, blocks):
    """The table of the larger tiles and of the grouped layouts, at the longest K it takes and one block beyond: the bits of the
    scales fetched through the re-layout pre-pass."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_contiguous, m_grouped_fp8_gemm_nt_masked
    print(f'case scale table {layout} {variant} {rows}x{N} {blocks} blocks', flush=True)
    G, K = 3, 128 * blocks
    a_q, a_s, b_q, b_s = helpers.make_dense(rows * (G if layout == 'masked' else 1), N if layout == 'dense' else 640 * G, K, seed=37)
    outs = []
    for knob in (0, 2):
        try:
            _lib.tune('scale_table', knob)
            if layout == 'dense':
                outs.append(_run_dense(dev, a_q, a_s, b_q, b_s, variant=variant))
                continue
            w = b_q.view(G, 640, K)[:, :N].contiguous().to(dev), b_s.view(G, 5, -1)[:, :-(-N // 128)].contiguous().to(dev)
            _lib.force_variant(variant)
            if layout == 'masked':
                valid = torch.tensor([rows, 1, rows - 37], dtype=torch.int32)
                out = torch.zeros(G, rows, N, dtype=torch.bfloat16, device=dev)
                m_grouped_fp8_gemm_nt_masked((a_q.view(G, rows, K).to(dev), a_s.view(G, rows, -1).to(dev)), w, out, valid.to(dev), rows)
            else:
                expert = torch.arange(rows, dtype=torch.int32) // 128 % G
                out = torch.zeros(rows, N, dtype=torch.bfloat16, device=dev)
                m_grouped_fp8_gemm_nt_contiguous((a_q.to(dev), a_s.to(dev)), w, out, expert.to(dev))
            torch.cuda.synchronize()
            outs.append(out)
        finally:
            _lib.tune('scale_table', 0)
            _lib.force_variant(None)
    assert torch.equal(outs[0], outs[1])
    if layout == 'dense':
        helpers.tolerance_check(outs[0], orc.dequant_ref(a_q, a_s, b_q, b_s), f'{layout} {variant}')
    else:
        last = outs[0].view(-1, rows, N)[-1][:1 if layout == 'masked' else rows].cpu()
        row = slice(2 * rows, 2 * rows + 1) if layout == 'masked' else slice(0, 128)
        ref = orc.dequant_ref(a_q[row], a_s[row], *(t.cpu() for t in ((w[0][2], w[1][2]) if layout == 'masked' else (w[0][0], w[1][0]))))
        helpers.tolerance_check(last[:ref.size(0)], ref, f'{layout} {variant}')


@pytest.mark.parametrize('variant,M', [('pipe256x256', 260), ('pipe128x256w8', 132)])
@pytest.mark.parametrize('kb,dtype', [(1, torch.bfloat16), (2, torch.float32), (3, torch.bfloat16), (4, torch.float32), (5, torch.float32),
                                      (15, torch.bfloat16), (16, torch.float32), (17, torch.bfloat16), (27, torch.bfloat16), (28, torch.float32)])
def test_tiles_of_a_resident_workgroup(dev, variant, M, kb, dtype):
    """258 tiles of 256 columns on 256 resident workgroups or fewer: the ring runs on into the next tile from as many K blocks
    on as it has stages; a last row tile of 4 rows and a last column tile of 233 columns, so that a workgroup goes from a
    whole tile to a ragged one; K on both sides of the longest whose scales come from the table (27 and 16 blocks)."""
    N, K = 33001, kb * 128
    print(f'case resident tiles {variant} K={K} {dtype}', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(M, N, K, seed=kb)
    outs = [_run_dense(dev, a_q, a_s, b_q, b_s, dtype=dtype, variant=variant) for _ in range(2)]
    assert torch.equal(outs[0], outs[1])
    helpers.tolerance_check(outs[0], orc.dequant_ref(a_q, a_s, b_q, b_s), f'resident tiles {variant} K={K}')


@pytest.mark.parametrize('variant,M,kb', [('pipe256x256', 2052, kb) for kb in (2, 3, 5, 28)] + [('pipe128x256w8', 1028, kb) for kb in (3, 4, 5, 17)] +
                         [('pipe128x128', 1028, kb) for kb in (3, 4, 5, 54, 55)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
def test_ring_runs_on_through_three_tiles(dev, variant, M, kb, dtype):
    """9 x 87 tiles of 256 columns or 9 x 73 of 128 on 256 workgroups, the last ones 4 rows high and 84 columns wide: tiles that start
    from a carried ring and carry it on, at as many K blocks as the ring has stages, one more, and counts that are no multiple of them,
    with the scale table (up to 27 / 16 / 54 blocks) and without.  The bits of the same kernel whose tiles start with an empty ring, which
    the knob asks for."""
    from dlblas_amd import _lib
    N, K = 9300 if variant == 'pipe128x128' else 22100, kb * 128
    print(f'case three tiles {variant} K={K} {dtype}', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(M, N, K, seed=kb)
    carried = _run_dense(dev, a_q, a_s, b_q, b_s, dtype=dtype, variant=variant)
    try:
        _lib.tune('epilogue', 2)
        apart = _run_dense(dev, a_q, a_s, b_q, b_s, dtype=dtype, variant=variant)
    finally:
        _lib.tune('epilogue', 0)
    assert torch.equal(carried, apart)
    rows = torch.tensor([0, 127, 128, 255, 256, 770, 1023, 1024, M - 1])
    helpers.tolerance_check(carried[rows.to(carried.device)], orc.dequant_ref(a_q[rows], a_s[rows], b_q, b_s), f'three tiles {variant} K={K}')


def test_refused_launch_enqueues_nothing(dev):
    """A call whose main kernel cannot be launched (here: a forced request for more LDS than the GPU has) returns
    DLB_ERR_LAUNCH before any pre-pass is enqueued: workspace and output keep their bytes."""
    import ctypes
    from dlblas_amd import _lib
    lib = _lib.load()
    M, N, K = 2048, 4096, 512  # row-major scales that are not to come through the table in LDS: the call starts with a re-layout pass
    a_q, a_s, b_q, b_s = (t.to(dev) for t in helpers.make_dense(M, N, K, seed=5))
    out = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=dev)
    ws = torch.full((_lib.WORKSPACE_BYTES, ), 0x5a, dtype=torch.uint8, device=dev)
    ws[:_lib.WS_COUNTER_BYTES] = 0
    vp = ctypes.c_void_p
    args = (vp(a_q.data_ptr()), vp(b_q.data_ptr()), vp(a_s.data_ptr()), vp(b_s.data_ptr()), vp(out.data_ptr()), M, N, K, a_s.stride(0),
            a_s.stride(1), _lib.OUT_BF16, vp(ws.data_ptr()), ws.numel(), vp(torch.cuda.current_stream().cuda_stream))
    try:
        _lib.tune('scale_table', 2)
        _lib.tune('lds_oversize', 1)
        rc = lib.dlb_fp8_gemm(*args)
        _lib.tune('lds_oversize', 0)
        torch.cuda.synchronize()
        assert rc == _lib.ERR_LAUNCH and 'nothing enqueued' in _lib.last_error()
        assert bool((ws[_lib.WS_COUNTER_BYTES:] == 0x5a).all()) and bool((out == 7.0).all())
        assert lib.dlb_fp8_gemm(*args) == 0  # the same call goes through once the hook is off ...
    finally:
        _lib.tune('lds_oversize', 0)
        _lib.tune('scale_table', 0)
    torch.cuda.synchronize()
    assert not bool((ws[_lib.WS_COUNTER_BYTES:] == 0x5a).all())  # ... and it does use the workspace
    helpers.tolerance_check(out, orc.dequant_ref(a_q.cpu(), a_s.cpu(), b_q.cpu(), b_s.cpu()), 'after a refused launch')


@pytest.mark.parametrize('M,N,K', [(2048, 4096, 512), (1000, 8192, 384), (2048, 8192, 256), (2048, 4096, 128), (200, 30000, 512)])
def test_short_k_takes_its_scales_from_the_table(dev, M, N, K):
    """One to four K blocks in the 128 x 256 tiles the planner picks there: no launch in front of the GEMM, so the workspace keeps
    its bytes; the bits of scales fetched through the re-layout pass."""
    import ctypes

    from dlblas_amd import _lib
    print(f'case short K {M}x{N}x{K}', flush=True)
    assert _lib.plan(0, M, N, K)[:2] == ('pipe128x256w8', 1) and _lib.plan_wave_k(M, N, K) is None
    a_q, a_s, b_q, b_s = (t.to(dev) for t in helpers.make_dense(M, N, K, seed=43))
    vp, stream, outs = ctypes.c_void_p, torch.cuda.current_stream().cuda_stream, []
    for knob in (0, 2):
        out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        ws = torch.full((_lib.WORKSPACE_BYTES, ), 0x5a, dtype=torch.uint8, device=dev)
        ws[:_lib.WS_COUNTER_BYTES] = 0
        try:
            _lib.tune('scale_table', knob)
            rc = _lib.load().dlb_fp8_gemm(vp(a_q.data_ptr()), vp(b_q.data_ptr()), vp(a_s.data_ptr()), vp(b_s.data_ptr()), vp(out.data_ptr()), M, N, K,
                                          a_s.stride(0), a_s.stride(1), _lib.OUT_BF16, vp(ws.data_ptr()), ws.numel(), vp(stream))
        finally:
            _lib.tune('scale_table', 0)
        torch.cuda.synchronize()
        assert rc == 0
        assert bool((ws[_lib.WS_COUNTER_BYTES:] == 0x5a).all()) == (knob == 0 or K == 128)  # scales of one K block are never laid out again
        outs.append(out)
    assert torch.equal(*outs)
    helpers.tolerance_check(outs[0], orc.dequant_ref(*(t.cpu() for t in (a_q, a_s, b_q, b_s))), f'short K {M}x{N}x{K}')


@pytest.mark.parametrize('variant', ['pipe256x256', 'pipe128x256w8', 'pipe256mix', 'pipe128x128', 'pipe128x64'])
@pytest.mark.parametrize('M,N,K', [(200, 392, 2048), (513, 1032, 256)])
def test_epilogue_through_lds_equals_direct_stores(dev, variant, M, N, K):
    """bf16 results of the 128 x 64 kernel leave through an LDS transpose (whole rows per store instruction) or, by knob, straight from
    the accumulator registers; those of the ring kernels from the registers, after lanes have exchanged pieces: the same fp32
    values, the same rounding, the same bits."""
    from dlblas_amd import _lib
    print(f'case epilogue variant={variant} M={M} N={N} K={K}', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(M, N, K, seed=23)
    try:
        _lib.tune('epilogue', 2)
        direct = _run_dense(dev, a_q, a_s, b_q, b_s, variant=variant)
    finally:
        _lib.tune('epilogue', 0)
    staged = _run_dense(dev, a_q, a_s, b_q, b_s, variant='pipe128x64')
    assert torch.equal(direct, staged)
    helpers.tolerance_check(direct, orc.dequant_ref(a_q, a_s, b_q, b_s), f'epilogue {variant}')


@pytest.mark.parametrize('variant', ['pipe256x256', 'pipe128x256w8', 'pipe256mix', 'pipe128x128', 'pipe128x64', None])
@pytest.mark.parametrize('M,N,K', [(257, 389, 256), (130, 1, 128), (33, 1023, 384), (130, 264, 384), (5, 387, 512), (300, 514, 1040)])
@pytest.mark.parametrize('out_dtype', [torch.bfloat16, torch.float32])
def test_rows_at_any_alignment(dev, variant, M, N, K, out_dtype):
    """Results that start at an odd element and rows that do, bf16 and fp32, in every kernel family: nothing is written beside them, and
    the bits are those of the 128 x 64 kernel, whose rows pass through LDS (that kernel itself: of its stores straight from the
    registers; the planner's choice, which may add K in another order: of its own result at an even element)."""
    from dlblas_amd import _lib
    if variant is not None and K % 128 != 0:
        pytest.skip('the ring kernels take whole K blocks')
    print(f'case rows variant={variant} M={M} N={N} K={K} {out_dtype}', flush=True)
    ops = helpers.make_dense(M, N, K, seed=29)
    even = _run_dense_guarded(dev, *ops, dtype=out_dtype, variant=variant)
    odd = _run_dense_guarded(dev, *ops, dtype=out_dtype, variant=variant, first=1)
    assert torch.equal(even, odd)
    if variant is not None:
        try:
            _lib.tune('epilogue', 2 if variant == 'pipe128x64' else 0)
            other = _run_dense_guarded(dev, *ops, dtype=out_dtype, variant='pipe128x64', first=1)
        finally:
            _lib.tune('epilogue', 0)
        assert torch.equal(even, other)
    helpers.tolerance_check(odd, orc.dequant_ref(*ops), f'rows {variant}')


@pytest.mark.parametrize('N', [389, 131, 514])
@pytest.mark.parametrize('variant', ['pipe256x256', 'pipe128x256w8', 'pipe128x128', 'tile128x128', None])
@pytest.mark.parametrize('out_dtype', [torch.bfloat16, torch.float32])
def test_stores_end_with_the_row(dev, N, variant, out_dtype):
    """The last valid row of an expert is followed by a row nobody may write: a store past the end of an odd row would show."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_masked
    G, cap, K = 3, 70, 256
    a_q, a_s, b_q, b_s = helpers.make_dense(G * cap, G * 640, K, seed=31)
    b_q = b_q.view(G, 640, K)[:, :N].contiguous()
    b_s = b_s.view(G, 5, -1)[:, :-(-N // 128)].contiguous()
    masked = torch.tensor([1, 33, 70], dtype=torch.int32)
    out = torch.full((G, cap, N), 7.0, dtype=out_dtype, device=dev)
    print(f'case row ends N={N} variant={variant} {out_dtype}', flush=True)
    try:
        _lib.force_variant(variant)
        m_grouped_fp8_gemm_nt_masked((a_q.view(G, cap, K).to(dev), a_s.view(G, cap, -1).to(dev)), (b_q.to(dev), b_s.to(dev)), out, masked.to(dev), 35)
        torch.cuda.synchronize()
    finally:
        _lib.force_variant(None)
    for g in range(G):
        v = int(masked[g])
        rows = slice(g * cap, g * cap + v)
        helpers.tolerance_check(out[g, :v].cpu(), orc.dequant_ref(a_q[rows], a_s[rows], b_q[g], b_s[g]), f'expert {g}')
        assert bool((out[g, v:] == 7.0).all())


@pytest.mark.parametrize('out_dtype', [torch.bfloat16, torch.float32])
@pytest.mark.parametrize('bn', [0, 4, 12, 20, 28, 32])
@pytest.mark.parametrize('M,N,K', [(16, 1000, 1024), (5, 130, 256), (40, 2112, 1024), (100, 392, 512)])
def test_decode_column_split(dev, M, N, K, bn, out_dtype):
    """Decode kernels with every width of the per-workgroup column range: ranges that are no multiple of 16 straddle
    weight-scale blocks (128 columns) inside a fragment and end in partly owned fragments; N itself is ragged."""
    from dlblas_amd import _lib
    print(f'case decode column split M={M} N={N} K={K} bn={bn} {out_dtype}', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(M, N, K, seed=31)
    ref = orc.dequant_ref(a_q, a_s, b_q, b_s)
    _lib.tune('skinny_bn', bn)
    _lib.tune('wave_k', 1)  # 40 and 100 rows
    try:
        out = _run_dense(dev, a_q, a_s, b_q, b_s, dtype=out_dtype)
    finally:
        _lib.tune('skinny_bn', 0)
        _lib.tune('wave_k', 0)
    assert out.dtype == out_dtype and tuple(out.shape) == (M, N)
    helpers.tolerance_check(out, ref, f'decode bn={bn} {M}x{N}x{K}')


@pytest.mark.parametrize('ws_bytes', [0, 65536 + 4096])
@pytest.mark.parametrize('M,N,K', [(128, 2112, 7168), (300, 2112, 1536), (16, 512, 1024)])
def test_c_abi_without_a_usable_workspace(dev, M, N, K, ws_bytes):
    """Straight through the C ABI with no workspace or one too small for anything: no re-laid scales, no K split,
    the same results."""
    import ctypes
    from dlblas_amd import _lib
    print(f'case no workspace M={M} N={N} K={K} ws_bytes={ws_bytes}', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(M, N, K, seed=17)
    ref = orc.dequant_ref(a_q, a_s, b_q, b_s)
    a, b, sa, sb = a_q.to(dev), b_q.to(dev), a_s.to(dev), b_s.to(dev)
    out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=dev)
    vp = ctypes.c_void_p
    rc = _lib.load().dlb_fp8_gemm(vp(a.data_ptr()), vp(b.data_ptr()), vp(sa.data_ptr()), vp(sb.data_ptr()), vp(out.data_ptr()),
                                  M, N, K, sa.stride(0), sa.stride(1), _lib.OUT_BF16, vp(ws.data_ptr() if ws_bytes else 0), ws_bytes,
                                  vp(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, _lib.last_error()
    torch.cuda.synchronize()
    helpers.tolerance_check(out, ref, f'no workspace {M}x{N}x{K}')


@pytest.mark.parametrize('M,N,K', [(0, 512, 1024), (16, 0, 1024), (16, 512, 0), (300, 392, 0)])
def test_empty_dimensions(dev, M, N, K):
    """No rows or no columns: an empty result; no K: a sum over nothing, i.e. zeros."""
    from dlblas_amd.kernels.fp8_gemm import fp8_gemm
    print(f'case empty M={M} N={N} K={K}', flush=True)
    a = torch.zeros(M, K, dtype=torch.uint8, device=dev).view(torch.float8_e4m3fn)
    b = torch.zeros(N, K, dtype=torch.uint8, device=dev).view(torch.float8_e4m3fn)
    a_s = torch.ones(M, (K + 127) // 128, device=dev)
    b_s = torch.ones((N + 127) // 128, (K + 127) // 128, device=dev)
    prev = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        out = fp8_gemm(a, b, a_s, b_s)
    finally:
        torch.set_default_dtype(prev)
    torch.cuda.synchronize()
    assert tuple(out.shape) == (M, N) and out.dtype == torch.bfloat16
    assert (out == 0).all()


def _random_shapes(n, seed):
    import random
    rng = random.Random(seed)
    shapes = []
    for _ in range(n):
        kind = rng.random()
        M = rng.choice([1, 2, 15, 16, 17, 31, 33, 64, 65, 127, 128, 129, 255, 257, 300, 511, 640])
        N = rng.choice([1, 7, 8, 24, 128, 130, 192, 200, 256, 264, 392, 520, 776, 1032])
        if kind < 0.6:
            K = 128 * rng.randint(1, 18)
        elif kind < 0.85:
            K = 16 * rng.randint(1, 60)
        else:
            K = rng.randint(1, 300)
        shapes.append((M, N, K))
    return shapes


@pytest.mark.parametrize('M,N,K', _random_shapes(40, 2024))
def test_dense_random_shapes_take_the_library_choice(dev, M, N, K):
    """Seeded random shapes across every branch of the shape heuristic (decode, split-K, pipelined, mixed, tiled with
    K tails, exact), bf16 and fp32 alternating."""
    out_dtype = torch.float32 if (M + N + K) % 2 else torch.bfloat16
    print(f'case random M={M} N={N} K={K} {out_dtype}', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(M, N, K, seed=M * 7 + N * 3 + K)
    out = _run_dense(dev, a_q, a_s, b_q, b_s, dtype=out_dtype)
    assert out.dtype == out_dtype and tuple(out.shape) == (M, N)
    helpers.tolerance_check(out, orc.dequant_ref(a_q, a_s, b_q, b_s), f'random {M}x{N}x{K}')


def test_limits_of_the_launch_grid_and_of_the_lds(dev):
    """More rows than the second grid dimension holds on the exact path (rows run in a grid-stride loop), and a forced
    decode wave count that would not fit the LDS (clamped): both launch and give the right answer."""
    from dlblas_amd import _lib
    M, N, K = 262200, 8, 8
    g = helpers.gen(5)
    a_q = torch.randint(-4, 5, (M, K), generator=g).float().to(torch.float8_e4m3fn)
    b_q = torch.randint(-4, 5, (N, K), generator=g).float().to(torch.float8_e4m3fn)
    a_s, b_s = torch.rand(M, 1, generator=g) + 0.5, torch.rand(1, 1, generator=g) + 0.5
    print(f'case exact path M={M}', flush=True)
    out = _run_dense(dev, a_q, a_s, b_q, b_s, dtype=torch.float32)
    ref = (a_q.float() @ b_q.float().t()) * a_s * b_s
    torch.testing.assert_close(out.cpu(), ref, rtol=1e-6, atol=0)
    try:
        _lib.tune('skinny_waves', 16)
        print('case skinny128 with 16 waves asked for', flush=True)
        a_q, a_s, b_q, b_s = helpers.make_dense(128, 512, 2048, seed=6)
        out = _run_dense(dev, a_q, a_s, b_q, b_s, variant='skinny128')
        helpers.tolerance_check(out, orc.dequant_ref(a_q, a_s, b_q, b_s), 'skinny128, 16 waves asked for')
    finally:
        _lib.tune('skinny_waves', 0)


def test_dense_f32_reference_test_construction(dev):
    """The reference's own test: randn e4m3 operands, randn (signed) scales, fp32 out, atol 1e-1
    (tests/kernels/test_fp8_gemm.py:8-31,70-72)."""
    print('case dense f32 reference construction', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_raw(512, 512, 512)
    ref = orc.dequant_ref(a_q, a_s, b_q, b_s)
    out = _run_dense(dev, a_q, a_s, b_q, b_s, dtype=torch.float32)
    assert out.dtype == torch.float32
    torch.testing.assert_close(out.cpu(), ref, atol=1e-1, rtol=0)
    helpers.tolerance_check(out, ref, 'reference construction')


def test_dense_exact_small_integers(dev):
    """Operands holding small integers and unit scales: every partial sum is an integer below 2^24, so the fp32
    result is exact whatever the summation order - bit-exact comparison."""
    print('case dense exact integers', flush=True)
    g = helpers.gen(3)
    M, N, K = 48, 272, 640
    a = torch.randint(-4, 5, (M, K), generator=g).float()
    b = torch.randint(-4, 5, (N, K), generator=g).float()
    a_q, b_q = a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn)
    a_s, b_s = torch.ones(M, 5), torch.ones(3, 5)
    out = _run_dense(dev, a_q, a_s, b_q, b_s, dtype=torch.float32)
    assert torch.equal(out.cpu(), a @ b.t())


def test_leading_dims_are_flattened(dev):
    print('case leading dims', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(6 * 5, 256, 256, seed=11)
    ref = orc.dequant_ref(a_q, a_s, b_q, b_s)
    out = _run_dense(dev, a_q.reshape(6, 5, 256), a_s.reshape(6, 5, 2), b_q, b_s)
    assert tuple(out.shape) == (6, 5, 256)
    helpers.tolerance_check(out.reshape(30, 256), ref, 'leading dims')


def test_contiguity_asserts(dev):
    from dlblas_amd.kernels.fp8_gemm import fp8_gemm
    a_q, a_s, b_q, b_s = (t.to(dev) for t in helpers.make_dense(32, 256, 256))
    with pytest.raises(AssertionError, match='Input tensors must be contiguous'):
        fp8_gemm(a_q.t().contiguous().t(), b_q, a_s, b_s)
    with pytest.raises(AssertionError, match='Scaling factor tensors must be contiguous'):
        fp8_gemm(a_q, b_q, a_s.t().contiguous().t(), b_s)


def test_repeat_calls_are_deterministic(dev):
    """Split-K partials are added in split order by whichever workgroup arrives last: bit-identical reruns."""
    print('case determinism', flush=True)
    a_q, a_s, b_q, b_s = helpers.make_dense(16, 2112, 7168, seed=5)
    outs = [_run_dense(dev, a_q, a_s, b_q, b_s) for _ in range(3)]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    a_q, a_s, b_q, b_s = helpers.make_dense(128, 1024, 4096, seed=5)
    outs = [_run_dense(dev, a_q, a_s, b_q, b_s) for _ in range(3)]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


# ----------------------------------------------------------------------------------------------------------------
# grouped
# ----------------------------------------------------------------------------------------------------------------
def _make_grouped_weights(G, N, K, seed):
    g = helpers.gen(seed)
    w = (torch.randn(G, N, K, generator=g) * 0.02).to(torch.bfloat16)
    qs = [orc.quant_weight_128x128(w[i]) for i in range(G)]
    return torch.stack([q for q, _ in qs]), torch.stack([s for _, s in qs])


@pytest.mark.parametrize('col_major_scales', [False, True])
@pytest.mark.parametrize('out_dtype', [torch.bfloat16, torch.float32])
def test_grouped_contiguous(dev, col_major_scales, out_dtype):
    print(f'case contiguous col_major={col_major_scales} {out_dtype}', flush=True)
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_contiguous
    G, N, K = 4, 384, 512
    counts = [128, 0, 384, 256]  # padded per-expert spans, one expert empty
    M_sum = sum(counts)
    g = helpers.gen(9)
    a = torch.randn(M_sum, K, generator=g).to(torch.bfloat16)
    a_q, a_s = orc.quant_act_1x128(a)
    w_q, w_s = _make_grouped_weights(G, N, K, 10)
    m_indices = torch.cat([torch.full((c, ), e, dtype=torch.int32) for e, c in enumerate(counts)])
    m_indices[128:256] = -1  # one skipped block
    sentinel = 777.0
    ref = orc.grouped_contiguous_ref(a_q, a_s, w_q, w_s, torch.full((M_sum, N), sentinel), m_indices)

    a_s_dev = a_s.to(dev)
    if col_major_scales:  # the layout dlblas/kernels/quant_dequant.py:65-83 hands over
        pad = -(-M_sum // 4) * 4
        buf = torch.zeros(K // 128, pad, device=dev)
        buf[:, :M_sum] = a_s_dev.t()
        a_s_dev = buf.t()[:M_sum]
        assert not a_s_dev.is_contiguous()
    out = torch.full((M_sum, N), sentinel, dtype=out_dtype, device=dev)
    m_grouped_fp8_gemm_nt_contiguous([a_q.to(dev), a_s_dev], (w_q.to(dev), w_s.to(dev)), out, m_indices.to(dev))
    torch.cuda.synchronize()
    assert torch.all(out[128:256] == sentinel), 'skipped block was written'
    helpers.tolerance_check(out, ref, 'grouped contiguous')


@pytest.mark.parametrize('variant', [None, 'list', 'pipe128x256w8', 'tile128x128'])
def test_grouped_contiguous_run_lengths(dev, variant):
    """Runs of 1 to 5 blocks of 128 rows, skipped blocks between and inside runs, an expert that owns two separate
    runs, experts out of order.  'list' pairs blocks into 256-row tiles from a list built on the device (the library's
    own choice for batches of more than two rounds of tiles; a batch this small gets 128 x 128 tiles); forced variants
    take the uniform 128-row path.  All must agree with the oracle."""
    print(f'case contiguous run lengths variant={variant}', flush=True)
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_contiguous
    G, N, K = 5, 520, 384
    blocks = [3, 3, -1, 0, 0, 0, 0, 0, 2, -1, -1, 4, 4, 4, 3, 1, 1, -1]   # expert of every 128-row block
    M_sum = 128 * len(blocks)
    g = helpers.gen(19)
    a_q, a_s = orc.quant_act_1x128(torch.randn(M_sum, K, generator=g).to(torch.bfloat16))
    w_q, w_s = _make_grouped_weights(G, N, K, 20)
    m_indices = torch.tensor(blocks, dtype=torch.int32).repeat_interleave(128)
    sentinel = 321.0
    ref = orc.grouped_contiguous_ref(a_q, a_s, w_q, w_s, torch.full((M_sum, N), sentinel), m_indices)
    out = torch.full((M_sum, N), sentinel, dtype=torch.bfloat16, device=dev)
    try:
        if variant == 'list':
            _lib.tune('tile_list', 1)
            assert _lib.plan(1, M_sum, N, K)[0] == 'pipe128x256w8'
        else:
            _lib.force_variant(variant)
        m_grouped_fp8_gemm_nt_contiguous((a_q.to(dev), a_s.to(dev)), (w_q.to(dev), w_s.to(dev)), out, m_indices.to(dev))
        torch.cuda.synchronize()
    finally:
        _lib.force_variant(None)
        _lib.tune('tile_list', 0)
    skipped = (m_indices < 0)
    assert torch.all(out.cpu()[skipped] == sentinel), 'a skipped block was written'
    helpers.tolerance_check(out, ref, f'contiguous run lengths {variant}')


@pytest.mark.parametrize('kb,dtype', [(1, torch.bfloat16), (2, torch.float32), (3, torch.bfloat16), (4, torch.bfloat16), (5, torch.float32), (8, torch.bfloat16)])
def test_list_tiles_carry_the_ring(dev, kb, dtype):
    """Four tiles of every height (128, 192 and 256 rows) by 130 column tiles, the last of them 233 columns wide: each resident
    workgroup goes through two or three tiles of a list, at fewer K blocks than the ring has stages, as many, and more.  Every
    result has the bits of the uniform 128-row tiles."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_contiguous
    blocks, N, K = [1, 2, 3, 2, 1, 1, 3, 2, 2, 1], 129 * 256 + 233, kb * 128
    print(f'case list ring K={K} {dtype}', flush=True)
    G, M_sum = len(blocks), 128 * sum(blocks)
    g = torch.Generator(device=dev).manual_seed(40 + kb)
    a_q, a_s = helpers.quantise_act_device(torch.randn(M_sum, K, device=dev, generator=g).to(torch.bfloat16))
    w_q, w_s = helpers.expert_weights_device(G, N, K, dev, 41)
    m_indices = torch.repeat_interleave(torch.arange(G, dtype=torch.int32), torch.tensor(blocks) * 128).to(dev)
    outs = []
    try:
        for variant in (None, 'pipe128x256w8'):
            out = torch.full((M_sum, N), 7.0, dtype=dtype, device=dev)
            _lib.tune('tile_list', 1 if variant is None else 0)
            _lib.force_variant(variant)
            m_grouped_fp8_gemm_nt_contiguous((a_q, a_s), (w_q, w_s), out, m_indices)
            outs.append(out)
    finally:
        _lib.force_variant(None)
        _lib.tune('tile_list', 0)
    assert torch.equal(outs[0], outs[1])
    rows = torch.tensor([0, 383, 384, 767, 768])  # experts 0 to 2
    ref = torch.cat([orc.dequant_ref(a_q[r:r + 1].cpu(), a_s[r:r + 1].cpu(), w_q[e].cpu(), w_s[e].cpu()) for r, e in zip(rows.tolist(), (0, 1, 2, 2, 3))])
    helpers.tolerance_check(outs[0][rows.to(dev)], ref, f'list ring K={K}')


# blocks per expert, column tiles, rows in the last block, whole tiles (256 / 192 rows) that the last round runs as 64-row pieces
LIST_CUTS = [([3, 3, 1, 3], 39, 128, (0, 17)), ([1, 3], 91, 1, (0, 17)), ([1, 3], 91, 64, (0, 17)), ([1, 3], 91, 65, (0, 17)), ([2], 270, 1, (14, 0)),
             ([2], 270, 64, (14, 0)), ([2], 270, 65, (14, 0))]


@pytest.mark.parametrize('blocks,tiles_n,last,cut', LIST_CUTS)
@pytest.mark.parametrize('kb,dtype', [(1, torch.bfloat16), (3, torch.float32), (5, torch.bfloat16)])
def test_list_tiles_in_pieces(dev, blocks, tiles_n, last, cut, kb, dtype):
    """A last round of few tiles runs as 64-row pieces: of 192-row tiles (an odd number, so that a pair is divided) and of the one 256-row
    tile; a last block so short that its last piece would start behind the last row, and one row more.  The bits of the
    uniform 128-row tiles, and the rows behind the last one stay as they were."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_contiguous
    assert helpers.list_cut(blocks, tiles_n, torch.cuda.get_device_properties(dev).multi_processor_count) == cut
    G, M_sum, N, K = len(blocks), 128 * (sum(blocks) - 1) + last, 256 * tiles_n - 23, kb * 128
    print(f'case list pieces blocks={blocks} last={last} N={N} K={K} {dtype}', flush=True)
    g = torch.Generator(device=dev).manual_seed(80 + kb)
    a_q, a_s = helpers.quantise_act_device(torch.randn(M_sum, K, device=dev, generator=g).to(torch.bfloat16))
    w_q, w_s = helpers.expert_weights_device(G, N, K, dev, 81)
    m_indices = torch.repeat_interleave(torch.arange(G, dtype=torch.int32), torch.tensor(blocks) * 128)[:M_sum].contiguous().to(dev)
    outs = []
    try:
        for variant in (None, 'pipe128x256w8'):
            whole = torch.full((M_sum + 64, N), 7.0, dtype=dtype, device=dev)
            _lib.tune('tile_list', 1 if variant is None else 0)
            _lib.force_variant(variant)
            assert _lib.plan_grouped(1, M_sum, N, K, G) == ('pipe128x256w8', variant is None)
            m_grouped_fp8_gemm_nt_contiguous((a_q, a_s), (w_q, w_s), whole[:M_sum], m_indices)
            torch.cuda.synchronize()
            assert bool((whole[M_sum:] == 7.0).all()), 'a row behind the last one was written'
            outs.append(whole[:M_sum])
    finally:
        _lib.force_variant(None)
        _lib.tune('tile_list', 0)
    assert torch.equal(outs[0], outs[1])
    rows = torch.tensor([M_sum - 1])
    helpers.tolerance_check(outs[0][rows.to(dev)], orc.dequant_ref(a_q[rows.to(dev)].cpu(), a_s[rows.to(dev)].cpu(), w_q[G - 1].cpu(), w_s[G - 1].cpu()), f'list pieces K={K}')


def test_grouped_contiguous_many_blocks(dev):
    """700 blocks of 128 rows: the device-side tile list then works in chunks of several blocks per thread, and runs of
    1 to 7 blocks (256-row tiles, pairs of 192-row tiles for the odd ones, single 128-row tiles) cross the chunk
    boundaries in every way.  Skipped blocks in between; the last block is short."""
    print('case contiguous many blocks', flush=True)
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_contiguous
    G, N, K = 12, 256, 128
    g = helpers.gen(31)
    blocks = []
    while len(blocks) < 700:
        e = int(torch.randint(-1, G, (1, ), generator=g))
        blocks += [e] * int(torch.randint(1, 8, (1, ), generator=g))
    blocks = blocks[:700]
    M_sum = 128 * len(blocks) - 37
    a_q, a_s = orc.quant_act_1x128(torch.randn(M_sum, K, generator=g).to(torch.bfloat16))
    w_q, w_s = _make_grouped_weights(G, N, K, 32)
    m_indices = torch.tensor(blocks, dtype=torch.int32).repeat_interleave(128)[:M_sum].contiguous()
    sentinel = 99.0
    ref = orc.grouped_contiguous_ref(a_q, a_s, w_q, w_s, torch.full((M_sum, N), sentinel), m_indices)
    out = torch.full((M_sum, N), sentinel, dtype=torch.bfloat16, device=dev)
    try:
        _lib.tune('tile_list', 1)  # at so short a K the planner keeps to the uniform tiles
        assert _lib.plan_grouped(1, M_sum, N, K, G) == ('pipe128x256w8', True)
        m_grouped_fp8_gemm_nt_contiguous((a_q.to(dev), a_s.to(dev)), (w_q.to(dev), w_s.to(dev)), out, m_indices.to(dev))
        torch.cuda.synchronize()
    finally:
        _lib.tune('tile_list', 0)
    assert torch.all(out.cpu()[m_indices < 0] == sentinel), 'a skipped block was written'
    helpers.tolerance_check(out, ref, 'contiguous many blocks')


def test_grouped_masked(dev):
    print('case masked', flush=True)
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_masked
    G, M_max, N, K = 6, 256, 512, 384
    g = helpers.gen(12)
    masked_m = torch.tensor([0, 1, 256, 130, 77, 128], dtype=torch.int32)
    a = torch.randn(G, M_max, K, generator=g).to(torch.bfloat16)
    a_q, a_s = orc.quant_act_1x128(a)
    w_q, w_s = _make_grouped_weights(G, N, K, 13)
    # rows at or beyond masked_m hold NaN codes and NaN scales: they must never reach a valid output
    a_bits = a_q.view(torch.uint8).clone()
    for e in range(G):
        a_bits[e, int(masked_m[e]):] = 0x7F
        a_s[e, int(masked_m[e]):] = float('nan')
    a_q = a_bits.view(torch.float8_e4m3fn)
    sentinel = -555.0
    ref = orc.grouped_masked_ref(a_q, a_s, w_q, w_s, torch.full((G, M_max, N), sentinel), masked_m)
    out = torch.full((G, M_max, N), sentinel, dtype=torch.bfloat16, device=dev)
    m_grouped_fp8_gemm_nt_masked((a_q.to(dev), a_s.to(dev)), (w_q.to(dev), w_s.to(dev)), out, masked_m.to(dev), 0)
    torch.cuda.synchronize()
    for e in range(G):
        assert torch.all(out[e, int(masked_m[e]):] == sentinel), f'expert {e}: rows beyond masked_m were written'
    assert not torch.isnan(out.float()).any()
    helpers.tolerance_check(out, ref, 'grouped masked')


def test_grouped_masked_hint_picks_the_tile_shape(dev):
    """expected_m picks the tile shape - unknown: 128 x 256; a few short experts: 128 x 128; several hundred rows per
    expert: 256-row tiles - and never a result bit."""
    print('case masked expected_m', flush=True)
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_masked
    G, M_max, N, K = 6, 512, 1536, 256
    g = helpers.gen(16)
    masked_m = torch.tensor([0, 1, 512, 130, 400, 257], dtype=torch.int32)
    a_q, a_s = orc.quant_act_1x128(torch.randn(G, M_max, K, generator=g).to(torch.bfloat16))
    w_q, w_s = _make_grouped_weights(G, N, K, 17)
    a_bits = a_q.view(torch.uint8).clone()
    for e in range(G):
        a_bits[e, int(masked_m[e]):] = 0x7F
        a_s[e, int(masked_m[e]):] = float('nan')
    a_q = a_bits.view(torch.float8_e4m3fn)
    sentinel = -555.0
    ref = orc.grouped_masked_ref(a_q, a_s, w_q, w_s, torch.full((G, M_max, N), sentinel), masked_m)
    outs, shapes = [], []
    for hint in (0, 16, 500):
        shapes.append(_lib.plan_grouped(2, M_max, N, K, G, hint)[0])
        out = torch.full((G, M_max, N), sentinel, dtype=torch.bfloat16, device=dev)
        m_grouped_fp8_gemm_nt_masked((a_q.to(dev), a_s.to(dev)), (w_q.to(dev), w_s.to(dev)), out, masked_m.to(dev), hint)
        torch.cuda.synchronize()
        for e in range(G):
            assert torch.all(out[e, int(masked_m[e]):] == sentinel), f'expected_m = {hint}, expert {e}: rows beyond masked_m were written'
        outs.append(out)
    assert shapes == ['pipe128x256w8', 'pipe128x128', 'pipe256x256'], shapes
    helpers.tolerance_check(outs[0], ref, 'masked expected_m')
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize('kb,dtype', [(1, torch.bfloat16), (2, torch.float32), (3, torch.bfloat16), (4, torch.float32), (5, torch.bfloat16), (17, torch.bfloat16)])
def test_masked_tiles_carry_the_ring(dev, kb, dtype):
    """Six experts of 0 to 300 rows by 25673 columns: every resident workgroup of the masked layout's ring kernels goes through several
    tiles, whole and ragged ones, of one expert and of the next, at fewer K blocks than the ring has stages, as many, and more
    (17: more than the scale table of the 128 x 256 tiles holds).  The three tile shapes and, from the three K blocks on that it needs,
    the weight-streaming kernel agree bit for bit, rows at or beyond masked_m stay as they were."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_masked
    G, M_max, N, K = 6, 300, 100 * 256 + 73, kb * 128
    print(f'case masked ring K={K} {dtype}', flush=True)
    g = torch.Generator(device=dev).manual_seed(50 + kb)
    masked_m = torch.tensor([300, 0, 1, 256, 129, 64], dtype=torch.int32)
    a_q, a_s = helpers.quantise_act_device(torch.randn(G * M_max, K, device=dev, generator=g).to(torch.bfloat16))
    a_q, a_s = a_q.view(G, M_max, K), a_s.view(G, M_max, kb)
    w_q, w_s = helpers.expert_weights_device(G, N, K, dev, 51)
    beyond = torch.arange(M_max)[None, :] >= masked_m[:, None]
    outs = []
    try:
        for variant in ('pipe256x256', 'pipe128x256w8', 'pipe128x128', 'stream128x256')[:3 if kb < 3 else 4]:
            out = torch.full((G, M_max, N), 7.0, dtype=dtype, device=dev)
            if variant == 'stream128x256':
                _lib.force_variant(None)
                _lib.tune('stream', 5)
                assert _lib.plan_stream(M_max, N, K, G, 150) == (128, 256, False)
            else:
                _lib.force_variant(variant)
            m_grouped_fp8_gemm_nt_masked((a_q, a_s), (w_q, w_s), out, masked_m.to(dev), 150)
            assert torch.all(out[beyond.to(dev)] == 7.0), f'{variant}: rows beyond masked_m were written'
            outs.append(out)
    finally:
        _lib.force_variant(None)
        _lib.tune('stream', 0)
    for out in outs[1:]:
        assert torch.equal(outs[0], out)
    for e, row in ((0, 299), (3, 255), (5, 0)):
        ref = orc.dequant_ref(a_q[e, row:row + 1].cpu(), a_s[e, row:row + 1].cpu(), w_q[e].cpu(), w_s[e].cpu())
        helpers.tolerance_check(outs[0][e, row:row + 1], ref, f'masked ring K={K} expert {e}')


@pytest.mark.parametrize('K', [384, 2048, 2176])
def test_grouped_masked_scale_table(dev, K):
    """The masked layout fetches a tile's row-major activation scales once, into a table in LDS, when K has at most 16
    blocks (no re-layout launch in front); longer K and the knob take the re-laid copy in the workspace.  Same bits
    either way, rows at or beyond masked_m (NaN codes, NaN scales) never read into a valid row nor written."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_masked
    print(f'case masked scale table K={K}', flush=True)
    G, M_max, N = 5, 256, 512
    g = helpers.gen(14)
    masked_m = torch.tensor([3, 256, 0, 129, 200], dtype=torch.int32)
    a_q, a_s = orc.quant_act_1x128(torch.randn(G, M_max, K, generator=g).to(torch.bfloat16))
    w_q, w_s = _make_grouped_weights(G, N, K, 15)
    a_bits = a_q.view(torch.uint8).clone()
    for e in range(G):
        a_bits[e, int(masked_m[e]):] = 0x7F
        a_s[e, int(masked_m[e]):] = float('nan')
    a_q = a_bits.view(torch.float8_e4m3fn)
    sentinel = -555.0
    ref = orc.grouped_masked_ref(a_q, a_s, w_q, w_s, torch.full((G, M_max, N), sentinel), masked_m)
    _lib.tune('stream', 1)  # the ring kernels
    outs = []
    for knob in (0, 2):
        out = torch.full((G, M_max, N), sentinel, dtype=torch.bfloat16, device=dev)
        _lib.tune('scale_table', knob)
        try:
            m_grouped_fp8_gemm_nt_masked((a_q.to(dev), a_s.to(dev)), (w_q.to(dev), w_s.to(dev)), out, masked_m.to(dev), 0)
            torch.cuda.synchronize()
        finally:
            _lib.tune('scale_table', 0)
        outs.append(out)
    _lib.tune('stream', 0)
    for e in range(G):
        assert torch.all(outs[0][e, int(masked_m[e]):] == sentinel)
    helpers.tolerance_check(outs[0], ref, f'masked scale table K={K}')
    assert torch.equal(outs[0], outs[1])


def test_registry_selects_and_caches_on_gpu(dev):
    print('case registry', flush=True)
    from dlblas_amd import get_op
    a_q, a_s, b_q, b_s = (t.to(dev) for t in helpers.make_dense(64, 512, 1024))
    op = get_op('fp8_gemm', (a_q, b_q, a_s, b_s))
    assert get_op('fp8_gemm', (a_q, b_q, a_s, b_s)) is op
    prev = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        out = op(a_q, b_q, a_s, b_s)
    finally:
        torch.set_default_dtype(prev)
    ref = orc.dequant_ref(a_q.cpu(), a_s.cpu(), b_q.cpu(), b_s.cpu())
    helpers.tolerance_check(out, ref, 'registry')


def test_registry_chooses_between_two_real_implementations(dev):
    """'fp8_gemm' has two registered implementations (the planner's kernels, the register-staged tile kernels): both
    match, both are benchmarked on the caller's tensors, the faster one is cached and returned, and both are right."""
    print('case registry selection', flush=True)
    from dlblas_amd import get_op
    from dlblas_amd.op_registry import op_registry
    from dlblas_amd.op_struct import match
    for (M, N, K) in ((16, 2112, 2048), (512, 1024, 2048)):
        a_q, a_s, b_q, b_s = (t.to(dev) for t in helpers.make_dense(M, N, K, seed=9))
        args = (a_q, b_q, a_s, b_s)
        cands = [impl for impl in op_registry.ops['fp8_gemm'] if match(args, impl.params)]
        assert len(cands) == 2 and cands[0].call is not cands[1].call
        ref = orc.dequant_ref(a_q.cpu(), a_s.cpu(), b_q.cpu(), b_s.cpu())
        prev = torch.get_default_dtype()
        torch.set_default_dtype(torch.bfloat16)
        try:
            op = get_op('fp8_gemm', args)
            assert op in cands and get_op('fp8_gemm', args) is op
            times = [min(impl.bench(*args) for _ in range(3)) for impl in cands]
            other = cands[1 - cands.index(op)]
            # the cached choice is the faster one (25 % slack: the two benches ran at different moments)
            assert times[cands.index(op)] <= 1.25 * times[cands.index(other)], (M, N, K, times)
            for impl in cands:
                helpers.tolerance_check(impl(*args), ref, f'registry candidate {impl.call.__name__} {M}x{N}x{K}')
        finally:
            torch.set_default_dtype(prev)
