"""The native form of the entry points (csrc/host_calls.cpp) does what their Python form does - same bits, same shapes and
strides - for the calls it takes, and leaves every other call to it."""
import threading

import pytest
import torch

import helpers
from oracle import fp8_block_gemm as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def dev():
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    return torch.device('cuda:0')


def _operands(lead, N, K, dev, seed=5):
    g = helpers.gen(seed)
    rows = 1
    for d in lead:
        rows *= d
    whole = -(-K // 128) * 128  # a ragged last block keeps the scale of the whole one
    a, a_s = orc.quant_act_1x128(torch.randn(rows, whole, generator=g).to(torch.bfloat16))
    b, b_s = orc.quant_weight_128x128((torch.randn(N, whole, generator=g) * 0.05).to(torch.bfloat16))
    a, b = a[:, :K].contiguous(), b[:, :K].contiguous()
    return a.view(*lead, K).to(dev), b.to(dev), a_s.view(*lead, -1).to(dev), b_s.to(dev)


@pytest.mark.parametrize('lead,N,K', [((1, ), 128, 256), ((3, 5), 136, 400), ((130, ), 512, 1024)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32, torch.float16])
def test_fp8_gemm_equals_the_custom_op(dev, lead, N, K, dtype):
    from dlblas_amd import _fast
    from dlblas_amd.kernels.fp8_gemm import fp8_gemm
    args = _operands(lead, N, K, dev)
    prev = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        native, out = _fast.fp8_gemm(*args), fp8_gemm(*args)
    finally:
        torch.set_default_dtype(prev)
    ref = torch.ops.dlblas.fp8_gemm(*args, dtype)
    torch.cuda.synchronize()
    assert (native is None) == (dtype == torch.float16)  # a type the kernels do not write is converted on the Python path
    assert out.dtype == ref.dtype and out.shape == ref.shape and torch.equal(out, ref)


@pytest.mark.parametrize('shape', [(7, 256), (2, 3, 384), (2, 1, 4, 128)])
@pytest.mark.parametrize('col_major', [False, True])
def test_quantiser_equals_the_custom_op(dev, shape, col_major):
    from dlblas_amd import _fast, _lib
    from dlblas_amd.kernels.fp8 import per_token_group_quant_fp8, quant_op
    x = torch.randn(*shape, generator=helpers.gen(6)).to(torch.bfloat16).to(dev)
    assert _fast.quant(x, 128, 1e-10, col_major) is not None
    q, s = per_token_group_quant_fp8(x, 128, column_major_scales=col_major)
    K = shape[-1]
    rows = x.numel() // K
    ref_q = torch.empty(rows, K, dtype=torch.float8_e4m3fn, device=dev)
    ref_s = torch.empty(rows, K // 128, device=dev)
    quant_op(x.view(-1, K), ref_q, ref_s, 1e-10, 128)
    torch.cuda.synchronize()
    assert q.shape == x.shape and torch.equal(q.view(-1, K).view(torch.uint8), ref_q.view(torch.uint8))
    assert s.shape == x.shape[:-1] + (K // 128, ) and torch.equal(s.reshape(rows, -1), ref_s)
    if col_major:
        buf = torch.empty((K // 128, ) + x.shape[:-1]).movedim(0, -1)
        assert s.stride() == buf.stride()
    wide = torch.randn(5, 512, device=dev)[:, :256]  # rows further apart than they are long
    assert torch.equal(per_token_group_quant_fp8(wide, 128)[1], per_token_group_quant_fp8(wide.contiguous(), 128)[1])


def test_other_calls_are_left_to_the_python_path(dev):
    from torch._subclasses.fake_tensor import FakeTensorMode

    from dlblas_amd import _fast
    from dlblas_amd.kernels.fp8_gemm import fp8_gemm
    a, b, a_s, b_s = _operands((16, ), 128, 256, dev)
    assert _fast.fp8_gemm(a, b, a_s, b_s) is not None
    assert _fast.fp8_gemm(a, b.t(), a_s, b_s) is None and _fast.fp8_gemm(a, b, a_s[:, :1], b_s) is None
    assert _fast.fp8_gemm(a, b, a_s, b_s.half()) is None and _fast.fp8_gemm(a, b, a_s.cpu(), b_s) is None
    assert _fast.fp8_gemm(a, b, a_s.clone().requires_grad_(), b_s) is None
    assert _fast.fp8_gemm(a, b, None, b_s) is None and _fast.fp8_gemm(a, b, torch.nn.Parameter(a_s), b_s) is None
    with FakeTensorMode() as mode:
        fake = [mode.from_tensor(t) for t in (a, b, a_s, b_s)]
        assert _fast.fp8_gemm(*fake) is None and tuple(fp8_gemm(*fake).shape) == (16, 128)

    class Calls(torch.overrides.TorchFunctionMode):
        seen = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Calls():
        fp8_gemm(a, b, a_s, b_s)
    assert any('dlblas.fp8_gemm' in f for f in Calls.seen)
    with pytest.raises(AssertionError, match='contiguous'):
        fp8_gemm(a[:, ::2], b, a_s, b_s)
    with pytest.raises(ValueError):
        fp8_gemm(a, b, a_s, b_s[:, :1].contiguous())


def test_streams_and_threads_share_the_workspaces_of_the_python_path(dev):
    """Partial sums of K slices lie in the workspace of (device, stream): threads on streams of their own, with operands of
    their own, would see each other's if two streams shared one."""
    from dlblas_amd import _fast, _lib
    from dlblas_amd.kernels.fp8_gemm import fp8_gemm
    M, N, K = 200, 392, 2048
    operands = [_operands((M, ), N, K, dev, seed=5 + i) for i in range(3)]
    _lib.tune('wave_k', 1)
    assert _lib.plan_wave_k(M, N, K) is None and _lib.plan(0, M, N, K)[1] > 1
    refs = [fp8_gemm(*args) for args in operands]
    torch.cuda.synchronize()
    assert not torch.equal(refs[0], refs[1])
    results, failed = {}, []

    def work(i):
        try:
            _lib.tune('wave_k', 1)  # knobs are the thread's own
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                assert _fast.fp8_gemm(*operands[i]) is not None
                outs = [fp8_gemm(*operands[i]) for _ in range(40)]
            stream.synchronize()
            results[i] = all(torch.equal(o, refs[i]) for o in outs)
            assert (dev.index or 0, stream.cuda_stream) in _lib._workspaces
        except Exception as exc:  # reported by the test's own thread
            failed.append(exc)

    threads = [threading.Thread(target=work, args=(i, )) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    assert len(results) == 3 and all(results.values())


@pytest.mark.parametrize('tokens,E', [(40, 3), (300, 2), (3000, 6)])
def test_fused_moe_v3_with_the_tile_lists_kept_equals_the_steps(dev, tokens, E):
    """The native expert MLP leaves the tile lists of the first GEMM to the second; under a function mode the Python path
    builds them for each.  Runs of 1, 2, 3 and more blocks per expert, an expert without rows, twice on one workspace."""
    from dlblas_amd import _fast, _lib
    from dlblas_amd.kernels.fp8 import per_block_quant_fp8, per_token_group_quant_fp8
    from dlblas_amd.kernels.fused_moe_v3 import fused_moe_v3
    H, inter = 512, 256
    g = helpers.gen(9)

    def weights(n, k):
        q, s = zip(*(per_block_quant_fp8((torch.randn(n, k, generator=g) * 0.05).to(torch.bfloat16).to(dev)) for _ in range(E)))
        return torch.stack(q), torch.stack(s)

    w13, w2 = weights(2 * inter, H), weights(H, inter)
    x = per_token_group_quant_fp8(torch.randn(tokens, H, generator=g).to(torch.bfloat16).to(dev), 128)
    share = torch.arange(1, E + 1).float()
    share[0] = 0
    try:
        for knob, value in (('tile_list', 1), ('stream', 1)):
            _lib.tune(knob, value)
        for _ in range(2):
            ids = torch.multinomial(share, 2 * tokens, replacement=True, generator=g).view(tokens, 2)
            counts = ((torch.bincount(ids.flatten(), minlength=E) + 127) // 128 * 128).tolist()
            args = ids.to(dev), torch.rand(tokens, 2, generator=g).to(dev), w13, w2, counts
            out = _fast.fused_moe_v3(*x, *args[:2], *w13, *w2, counts)
            with torch.overrides.BaseTorchFunctionMode():
                ref = fused_moe_v3(x, *args)
            torch.cuda.synchronize()
            assert out is not None and torch.equal(out, ref)
    finally:
        _lib.tune('tile_list', 0), _lib.tune('stream', 0)


@pytest.mark.parametrize('tokens,topk,E,H', [
    (4097, 8, 256, 256),     # one token more than 256 experts' histograms may have for counts in the launch
    (300, 4, 300, 256),      # more experts than counts travel in the launch
    (131073, 1, 2, 16384),   # token offsets of 32 bits: no row ranges (every fourth token is routed here)
])
def test_fused_moe_v3_reads_the_tokens_in_place_beyond_the_native_call(dev, monkeypatch, tokens, topk, E, H):
    """Batches that the native call leaves to the Python path still go through row tables and the gathering GEMM, with no
    expert-sorted copy of the activations, and give the bits of the three steps."""
    import importlib

    from dlblas_amd import _fast, _lib
    moe = importlib.import_module('dlblas_amd.kernels.fused_moe_v3')
    print(f'case fused_moe_v3 in place tokens={tokens} topk={topk} E={E} H={H}', flush=True)
    inter = 128
    g = torch.Generator(device=dev).manual_seed(12)

    def codes(*shape):  # finite e4m3 codes of either sign
        return (torch.randint(0, 0x60, shape, device=dev, generator=g, dtype=torch.uint8) |
                (torch.randint(0, 2, shape, device=dev, generator=g, dtype=torch.uint8) << 7)).view(torch.float8_e4m3fn)

    def scales(*shape):
        return torch.rand(*shape, device=dev, generator=g) * 2e-3 + 1e-3

    x = codes(tokens, H), scales(tokens, H // 128)
    w13, w2 = (codes(E, 2 * inter, H), scales(E, 2, H // 128)), (codes(E, H, inter), scales(E, H // 128, 1))
    ids = torch.randint(0, E, (tokens, topk), device=dev, generator=g)
    if tokens > 100000:
        ids[torch.arange(tokens, device=dev) % 4 > 0] = -1
    wts = torch.rand(tokens, topk, device=dev, generator=g)
    counts = ((torch.bincount(ids[ids >= 0], minlength=E) + 127) // 128 * 128).tolist()
    ran = []
    copy, tables, gemm = moe.ep_scatter, moe.ep_scatter_rows, moe.fp8_gemm_grouped_contiguous_silu_quant
    monkeypatch.setattr(moe, 'ep_scatter', lambda *a: (ran.append('copy'), copy(*a)))
    monkeypatch.setattr(moe, 'ep_scatter_rows', lambda *a: (ran.append('tables'), tables(*a)))
    monkeypatch.setattr(moe, 'fp8_gemm_grouped_contiguous_silu_quant',
                        lambda *a, **kw: (ran.append('gathering GEMM' if 'a_row_index' in kw else 'GEMM'), gemm(*a, **kw))[1])
    _lib.tune('stream', 1), _lib.tune('tile_list', 1)
    assert _fast.fused_moe_v3(*x, ids, wts, *w13, *w2, counts) is None
    out = moe.fused_moe_v3(x, ids, wts, w13, w2, counts)
    assert 'gathering GEMM' in ran and 'copy' not in ran
    assert ('tables' in ran) == (H == 256)  # the last one's counts do travel in the launch
    del ran[:]
    _lib.tune('tile_list', 2)
    ref = moe.fused_moe_v3(x, ids, wts, w13, w2, counts)
    torch.cuda.synchronize()
    assert ran == ['copy']  # ... and three steps
    assert torch.equal(out, ref) and bool(out.isfinite().all()) and float(out.abs().max()) > 0


def _small_experts(dev, E=2, H=512, inter=512):
    g = torch.Generator(device=dev).manual_seed(5)
    codes = lambda *s: torch.randint(0, 0x60, s, device=dev, generator=g, dtype=torch.uint8).view(torch.float8_e4m3fn)
    return (codes(E, 2 * inter, H), torch.ones(E, 2 * inter // 128, H // 128, device=dev)), (codes(E, H, inter), torch.ones(E, H // 128, inter // 128, device=dev)), codes


@pytest.mark.parametrize('inter,down_form', [(256, 'ON_WHOLE_BLOCKS'), (512, 'ON_ROW_RANGES')])
def test_fused_moe_v3_on_its_python_path_under_a_16_bit_default_dtype(dev, inter, down_form):
    """The default dtype is the type fp8_gemm returns; it changes no scale and no bit of an expert MLP, in either order of the scales
    between its GEMMs."""
    from dlblas_amd import _fast, _lib
    from dlblas_amd.kernels.fused_moe_v3 import fused_moe_v3
    H, T = 512, 40
    w13, w2, codes = _small_experts(dev, 2, H, inter)
    x = codes(T, H), torch.full((T, H // 128), 2e-3, device=dev)
    ids = (torch.arange(2 * T, device=dev) % 2).view(T, 2)
    wts, counts = torch.ones(T, 2, device=dev), [128, 128]
    plan = lambda n, k, quantising: _lib.expert_plan(1, 256, n, k, 2, 40, quantising)
    assert (plan(2 * inter, H, True), plan(H, inter, False)) == (_lib.ON_ROW_RANGES, getattr(_lib, down_form))
    print(f'case 16-bit default dtype {down_form}', flush=True)
    ref = _fast.fused_moe_v3(*x, ids, wts, *w13, *w2, counts)
    prev = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.overrides.BaseTorchFunctionMode():
            out = fused_moe_v3(x, ids, wts, w13, w2, counts)
    finally:
        torch.set_default_dtype(prev)
    torch.cuda.synchronize()
    assert torch.equal(out, ref) and bool(out.isfinite().all()) and float(out.abs().max()) > 0


def test_native_calls_are_ops_to_the_profiler(dev):
    """Every native call leaves an op event, with its inputs' shapes where they are asked for."""
    from dlblas_amd.kernels.fp8 import per_token_group_quant_fp8
    from dlblas_amd.kernels.fp8_gemm import fp8_gemm
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_contiguous, m_grouped_fp8_gemm_nt_masked
    from dlblas_amd.kernels.fused_moe_v3 import ep_gather, fused_moe_v3
    from dlblas_amd.kernels.moe import low_latency_experts
    w13, w2, codes = _small_experts(dev)
    args = _operands((16, ), 128, 256, dev)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=dev)
    a3, s3 = codes(2, 64, 512), torch.ones(2, 64, 4, device=dev)
    ids, wts = torch.tensor([[0], [1], [0]], device=dev), torch.ones(3, 1, device=dev)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], record_shapes=True) as prof:
        per_token_group_quant_fp8(torch.ones(4, 256, dtype=torch.bfloat16, device=dev), 128)
        fp8_gemm(*args)
        m_grouped_fp8_gemm_nt_contiguous((codes(128, 512), torch.ones(128, 4, device=dev)), w13, torch.empty(128, 1024, dtype=torch.bfloat16, device=dev),
                                         torch.zeros(128, dtype=torch.int32, device=dev))
        m_grouped_fp8_gemm_nt_masked((a3, s3), w13, torch.empty(2, 64, 1024, dtype=torch.bfloat16, device=dev), i32(3, 0), 2)
        down = low_latency_experts((a3, s3), *w13, *w2, i32(3, 1), 2)
        ep_gather(down.view(-1, 512), ids, wts, i32(0, 64, 1).view(3, 1), torch.empty(3, 512, dtype=torch.bfloat16, device=dev))
        fused_moe_v3((codes(3, 512), torch.ones(3, 4, device=dev)), ids, wts, w13, w2, [128, 128])
        torch.cuda.synchronize()
    shapes = {e.name: e.input_shapes for e in prof.events() if e.name.startswith('dlblas::')}
    assert shapes.keys() >= {'dlblas::' + n for n in ('per_token_group_quant_fp8', 'fp8_gemm', 'fp8_gemm_grouped_contiguous', 'fp8_gemm_grouped_masked',
                                                      'low_latency_experts', 'ep_gather', 'fused_moe_v3')}
    assert shapes['dlblas::fp8_gemm'][:2] == [[16, 256], [128, 256]]


def test_tensors_with_a_tangent_are_left_to_the_python_path(dev):
    """Forward-mode derivatives are the dispatcher's to refuse or to drop, not the native call's to overlook."""
    from torch.autograd import forward_ad

    from dlblas_amd import _fast
    x = torch.randn(4, 256, device=dev)
    assert _fast.quant(x, 128, 1e-10, False) is not None
    with forward_ad.dual_level():
        assert _fast.quant(forward_ad.make_dual(x, torch.ones_like(x)), 128, 1e-10, False) is None
    assert _fast.quant(x, 128, 1e-10, False) is not None


def _calls_through_the_workspace(dev):
    """name -> a call whose launches hand data on in the workspace: K slices, tile lists with re-laid scales, histograms."""
    from dlblas_amd.kernels.fp8_gemm import fp8_gemm
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_contiguous
    from dlblas_amd.kernels.fused_moe_v3 import ep_scatter_rows
    w13, _, codes = _small_experts(dev)
    args = _operands((200, ), 392, 2048, dev)
    a, a_s, idx = codes(512, 512), torch.ones(512, 4, device=dev), torch.zeros(512, dtype=torch.int32, device=dev)
    i32 = lambda n: torch.empty(n, dtype=torch.int32, device=dev)
    ids = torch.zeros(4000, 8, dtype=torch.int64, device=dev)
    return {
        'native dense': lambda: fp8_gemm(*args),
        'custom op dense': lambda: torch.ops.dlblas.fp8_gemm(*args, torch.bfloat16),
        'native contiguous': lambda: m_grouped_fp8_gemm_nt_contiguous((a, a_s), w13, torch.empty(512, 1024, dtype=torch.bfloat16, device=dev), idx),
        'row tables': lambda: ep_scatter_rows(ids, torch.tensor([32000, 0], dtype=torch.int32, device=dev), i32(2), i32(32000), i32(32000),
                                              torch.empty_like(ids)),
    }


@pytest.mark.parametrize('name', ['native dense', 'custom op dense', 'native contiguous', 'row tables'])
def test_launches_of_a_call_go_out_under_the_lock_of_its_workspace(dev, name):
    """Two threads on one stream share its workspace: a call waits while another one's launches are being enqueued."""
    import ctypes

    from dlblas_amd import _lib
    lib = _lib.load()
    call = _calls_through_the_workspace(dev)[name]
    call()
    torch.cuda.synchronize()
    ws = ctypes.c_void_p(_lib.workspace(dev, torch.cuda.current_stream().cuda_stream).data_ptr())
    done = threading.Event()

    def work():
        call()
        done.set()

    assert lib.dlb_workspace_lock(ws) == 0 and lib.dlb_workspace_lock(ws) == 0
    worker = threading.Thread(target=work)
    try:
        call()  # the holder's own calls go on
        worker.start()
        assert not done.wait(0.3)
    finally:
        lib.dlb_workspace_unlock(ws), lib.dlb_workspace_unlock(ws)
    assert done.wait(20)
    worker.join()
    torch.cuda.synchronize()


def test_native_calls_run_without_the_interpreter_lock(dev):
    """A launch waits while the hardware queue is full; other Python threads go on meanwhile.  PyGILState_Check stands in for
    the library's launching entry points: it returns 0, which is success to the caller, when the lock is not held."""
    import ctypes

    from dlblas_amd import _fast, _lib
    lib = _lib.load()
    w13, w2, codes = _small_experts(dev)
    args = _operands((16, ), 128, 256, dev)
    a3, s3, mm = codes(2, 64, 512), torch.ones(2, 64, 4, device=dev), torch.tensor([3, 0], dtype=torch.int32, device=dev)
    ids, wts = torch.tensor([[0], [1], [0]], device=dev), torch.ones(3, 1, device=dev)
    calls = {
        'fp8_gemm': args, 'quant': (torch.ones(4, 256, device=dev), 128, 1e-10, False),
        'grouped_contiguous': (codes(128, 512), torch.ones(128, 4, device=dev), *w13, torch.empty(128, 1024, device=dev), torch.zeros(128, dtype=torch.int32, device=dev)),
        'grouped_masked': (a3, s3, *w13, torch.empty(2, 64, 1024, device=dev), mm, 2),
        'low_latency_experts': (a3, s3, *w13, *w2, mm, 2),
        'ep_gather': (torch.ones(4, 512, device=dev), ids, wts, ids, torch.empty(3, 512, device=dev)),
        'fused_moe_v3': (codes(3, 512), torch.ones(3, 4, device=dev), ids, wts, *w13, *w2, [128, 128]),
    }
    assert calls.keys() == set(_fast._FUNCTIONS)
    # an expert MLP on row ranges (above), and one whose K is too short for them in the first and the second projection
    (v13, v2, _), form = _small_experts(dev, 2, 256, 256), lambda n, k, quantising: _lib.expert_plan(1, 256, n, k, 2, 2, quantising)
    assert (form(1024, 512, True), form(512, 512, False)) == (_lib.ON_ROW_RANGES, _lib.ON_ROW_RANGES)
    assert (form(512, 256, True), form(256, 256, False)) == (_lib.ON_WHOLE_BLOCKS, _lib.ON_WHOLE_BLOCKS)
    calls = list(calls.items()) + [('fused_moe_v3', (codes(3, 256), torch.ones(3, 2, device=dev), ids, wts, *v13, *v2, [128, 128]))]
    for name, a in calls:  # with the library itself: nothing declines these
        assert getattr(_fast, name)(*a) is not None, name
    torch.cuda.synchronize()
    init = _fast.fp8_gemm.__self__.init
    address = lambda f: ctypes.cast(f, ctypes.c_void_p).value
    real = [address(getattr(lib, n)) for n in _fast._ABI]
    asks = ('dlb_last_error', 'dlb_workspace_lock', 'dlb_workspace_unlock', 'dlb_expert_plan', 'dlb_ep_scatter_workspace_bytes')
    assert set(asks) <= set(_fast._ABI)
    probe = address(ctypes.pythonapi.PyGILState_Check)
    try:
        init([r if n in asks else probe for n, r in zip(_fast._ABI, real)], _lib.workspace)
        without = [(name, getattr(_fast, name)(*a) is not None) for name, a in calls]
    finally:
        init(real, _lib.workspace)
    assert all(went for _, went in without), without


def test_threads_on_one_stream_keep_their_launches_together(dev):
    """Threads that share a stream share its workspace: every call's partial sums are still its own."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm import fp8_gemm
    M, N, K = 200, 392, 2048
    operands = [_operands((M, ), N, K, dev, seed=5 + i) for i in range(3)]
    _lib.tune('wave_k', 1)
    refs = [fp8_gemm(*args) for args in operands]
    torch.cuda.synchronize()
    results = {}

    def work(i):
        _lib.tune('wave_k', 1)
        call = (lambda: fp8_gemm(*operands[i])) if i else (lambda: torch.ops.dlblas.fp8_gemm(*operands[i], torch.get_default_dtype()))
        outs = [call() for _ in range(100)]
        torch.cuda.synchronize()
        results[i] = all(torch.equal(o, refs[i]) for o in outs)

    threads = [threading.Thread(target=work, args=(i, )) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(results) == 3 and all(results.values())
