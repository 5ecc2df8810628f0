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
AHEAD = ['64x256 ahead', '64x128 ahead', '128x256 ahead', '64x64 ahead']  # knob values 8 .. 11


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
    ([40, 100], 100, 384, 256, torch.bfloat16, False),                  # 2 K blocks: shorter than every ring
    ([128, 64, 97], 128, 256, 384, torch.bfloat16, True),               # 3 K blocks: as short as the three-stage rings
    ([150, 256, 300, 129] * 5, 304, 2048, 1152, torch.bfloat16, False), # several tiles per workgroup, most of them full
    ([190, 70, 0, 33] * 6, 192, 1160, 2304, torch.float32, True),       # 18 blocks in two chunks; full and short tiles in turn
])
def test_masked_equals_the_ring_kernels(dev, masked, M_max, N, K, out_dtype, col_major):
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_masked
    a_q, a_s, w_q, w_s, mm = _inputs(masked, M_max, N, K, 40 + N + K, dev)
    if col_major:
        a_s = a_s.transpose(1, 2).contiguous().transpose(1, 2)
    outs = []
    for knob, shape in zip([1, 2, 3, 4, 5, 6, 8, 9, 10, 11], ['ring'] + SHAPES + AHEAD):
        print(f'case stream masked={masked[:6]} M_max={M_max} N={N} K={K} {out_dtype} shape={shape}', flush=True)
        out = torch.full((len(masked), M_max, N), -555.0, dtype=out_dtype, device=dev)
        _lib.tune('stream', knob)
        m_grouped_fp8_gemm_nt_masked((a_q, a_s), (w_q, w_s), out, mm, 0)
        torch.cuda.synchronize()
        _lib.tune('stream', 0)
        outs.append(out)
    for shape, out in zip(SHAPES + AHEAD, outs[1:]):
        assert torch.equal(out, outs[0]), shape
    ref = orc.grouped_masked_ref(a_q.cpu(), a_s.cpu(), w_q.cpu(), w_s.cpu(), torch.full((len(masked), M_max, N), -555.0), mm.cpu())
    valid = torch.arange(M_max)[None, :] < mm.cpu()[:, None]
    assert (outs[1].cpu()[~valid] == -555.0).all()
    if valid.any():
        helpers.tolerance_check(outs[1].cpu()[valid], ref[valid], f'stream {N}x{K}')


@pytest.mark.parametrize('masked,M_max,N,K', [([1, 63, 64, 0, 7], 64, 264, 1280), ([70, 128, 33] * 4, 128, 1024, 1152)])
def test_masked_results_at_an_odd_element(dev, masked, M_max, N, K):
    """The same bits where the results start on an element that is no dword: kernels that store through buffer descriptors leave
    such calls to plain stores."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_masked
    a_q, a_s, w_q, w_s, mm = _inputs(masked, M_max, N, K, 80 + N + K, dev)
    count = len(masked) * M_max * N
    for knob, shape in zip([2, 3, 4, 5, 6, 8, 9, 10, 11], SHAPES + AHEAD):
        outs = []
        for first in (0, 1):
            print(f'case stream masked={masked[:6]} M_max={M_max} N={N} K={K} shape={shape} first element {first}', flush=True)
            whole = torch.full((count + 8, ), -555.0, dtype=torch.bfloat16, device=dev)
            out = whole[first:first + count].view(len(masked), M_max, N)
            _lib.tune('stream', knob)
            m_grouped_fp8_gemm_nt_masked((a_q, a_s), (w_q, w_s), out, mm, 0)
            torch.cuda.synchronize()
            _lib.tune('stream', 0)
            assert (whole[:first] == -555.0).all() and (whole[first + count:] == -555.0).all()
            outs.append(out)
        assert torch.equal(outs[0], outs[1]), shape


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


@pytest.mark.parametrize('T,K,inter,E,topk,shape', [
    (96, 512, 256, 4, 2, '32x256'),
    (250, 1024, 384, 8, 4, '128x256'),    # up to two row tiles per expert
    (40, 2176, 128, 70, 3, '64x256'),     # experts without a token; a second window of experts
])
def test_ragged_rows_equal_the_contiguous_kernels(dev, T, K, inter, E, topk, shape):
    """Row ranges instead of m_indices, rows gathered through the token table: the bytes, scales and products of the
    expert-contiguous kernels on every row that holds a token; rows no range names keep their content."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import fp8_gemm_grouped_contiguous_silu_quant, m_grouped_fp8_gemm_nt_contiguous
    print(f'case ragged T={T} K={K} I={inter} E={E} topk={topk} {shape}', flush=True)
    g = helpers.gen(300 + T)
    x_q, x_s = orc.quant_act_1x128((torch.randn(T, K, generator=g) * 1.5).to(torch.bfloat16))
    quant = lambda n, k: [orc.quant_weight_128x128((torch.randn(n, k, generator=g) * 0.05).to(torch.bfloat16)) for _ in range(4)]
    stack = lambda ws: tuple(torch.stack([ws[e % 4][i] for e in range(E)]).to(dev) for i in (0, 1))
    (w13_q, w13_s), (w2_q, w2_s) = stack(quant(2 * inter, K)), stack(quant(256, inter))
    ids = torch.randint(-1, E, (T, topk), generator=g)
    routed = torch.bincount(ids[ids >= 0], minlength=E)
    counts = ((routed + 127) // 128 * 128).tolist()
    rows = sum(counts)
    i32 = lambda *s: torch.full(s, -9, dtype=torch.int32, device=dev)
    start, end, first, m_indices, row_token, slot = i32(E), i32(E), i32(E), i32(rows), i32(rows), torch.full_like(ids, -9, device=dev)
    assert _lib.ep_scatter_rows_host(ids.to(dev), counts, start, end, first, m_indices, row_token, slot)
    excl = torch.cumsum(torch.tensor([0] + counts[:-1]), 0)
    assert torch.equal(start.cpu().long(), excl) and torch.equal(end.cpu().long(), excl + routed) and torch.equal(first, end)
    x_q, x_s = x_q.to(dev), x_s.to(dev)
    ref_q, ref_s = fp8_gemm_grouped_contiguous_silu_quant(x_q, x_s, w13_q, w13_s, m_indices, a_row_index=row_token)
    _lib.tune('stream', 2 + SHAPES.index(shape))
    q = torch.full((rows, inter), 0x5a, dtype=torch.uint8, device=dev).view(torch.float8_e4m3fn)
    s = torch.full((rows, inter // 128), -7.0, device=dev)
    assert _lib.gemm_ragged_silu_quant(x_q, w13_q, x_s, w13_s, q, s, start, end, row_token, 64, 1e-10)
    sorted_q, sorted_s = x_q.view(torch.uint8)[row_token.long()].view(torch.float8_e4m3fn), x_s[row_token.long()]
    q2, s2 = torch.zeros_like(q), torch.zeros_like(s)
    assert _lib.gemm_ragged_silu_quant(sorted_q, w13_q, sorted_s, w13_s, q2, s2, start, end, None, 64, 1e-10)
    row = torch.arange(rows, device=dev)
    held = ((row[None] >= start[:, None]) & (row[None] < end[:, None])).any(0)
    torch.cuda.synchronize()
    for got_q, got_s in ((q, s), (q2, s2)):
        assert torch.equal(got_q.view(torch.uint8)[held], ref_q.view(torch.uint8)[held]) and torch.equal(got_s[held], ref_s[held])
    assert (s[~held] == -7.0).all() and (q.view(torch.uint8)[~held] == 0x5a).all()
    if inter % 256 == 0 or inter == 128 and shape != '128x256':
        out = torch.full((rows, 256), -555.0, dtype=torch.bfloat16, device=dev)
        if _lib.gemm_ragged(q, w2_q, s, w2_s, out, start, end, 64):
            ref = torch.zeros(rows, 256, dtype=torch.bfloat16, device=dev)
            m_grouped_fp8_gemm_nt_contiguous((ref_q, ref_s), (w2_q, w2_s), ref, m_indices)
            torch.cuda.synchronize()
            assert torch.equal(out[held], ref[held]) and (out[~held] == -555.0).all()


@pytest.mark.parametrize('T,topk,E', [(1, 1, 1), (33, 8, 32), (2048, 8, 32), (2049, 8, 300), (5000, 64, 7)])
def test_row_tables_around_the_one_launch_limit(dev, T, topk, E):
    """16384 entries are the most that one launch ranks by itself; expert counts that are no power of two; token counts
    that leave the last block short."""
    from dlblas_amd.kernels.fused_moe_v3 import ep_scatter_rows
    print(f'case row tables T={T} topk={topk} E={E}', flush=True)
    g = helpers.gen(T + E)
    ids = torch.randint(-2, E, (T, topk), generator=g)
    flat = ids.flatten()
    routed = torch.bincount(flat[flat >= 0], minlength=E)
    counts = (routed + 127) // 128 * 128
    rows = int(counts.sum())
    i32 = lambda n: torch.full((n, ), -9, dtype=torch.int32, device=dev)
    first, m_indices, src, slot = i32(E), i32(rows), i32(rows), torch.full_like(ids, -9, device=dev)
    ep_scatter_rows(ids.to(dev), counts.to(torch.int32).to(dev), first, m_indices, src, slot)
    torch.cuda.synchronize()
    excl = torch.cumsum(counts, 0) - counts
    order = torch.sort(flat, stable=True)
    rank = torch.empty_like(flat)
    n_none = int((flat < 0).sum())
    cum = torch.cumsum(routed, 0) - routed
    pos = torch.arange(flat.numel()) - n_none
    dest = torch.where(order.values >= 0, excl[order.values.clamp(min=0)] + pos - cum[order.values.clamp(min=0)], torch.full_like(pos, -9))
    rank[order.indices] = dest
    assert torch.equal(slot.cpu().flatten(), rank)
    assert torch.equal(first.cpu().long(), excl + routed)
    assert torch.equal(m_indices.cpu().long(), torch.repeat_interleave(torch.arange(E), counts))
    src_ref = torch.zeros(rows, dtype=torch.long)
    src_ref[rank[flat >= 0]] = (torch.arange(flat.numel()) // topk)[flat >= 0]
    assert torch.equal(src.cpu().long(), src_ref)


def _row_tables_ref(ids, counts):
    """Tables of the stable counting sort: first row of every expert, destination row of every slot (-9: none), token of
    every destination row (0 where no slot lies)."""
    flat = ids.flatten()
    excl = torch.cumsum(counts, 0) - counts
    routed = torch.bincount(flat[flat >= 0], minlength=len(counts))
    dest = torch.full_like(flat, -9)
    order = torch.sort(flat, stable=True).indices[int((flat < 0).sum()):]
    dest[order] = torch.cat([torch.arange(int(a), int(a) + int(n)) for a, n in zip(excl, routed)])
    return excl, routed, dest


@pytest.mark.parametrize('T,topk,E', [(33, 4, 5), (2100, 8, 40), (5000, 8, 300)])
def test_row_tables_longer_than_the_spans(dev, T, topk, E):
    """A table of fixed capacity: its rows past the experts' spans name token 0, whichever of the three forms of the kernel
    fills it (the ids ranked in one launch, summed histograms, scanned histograms), and keep the -1 that the caller put
    into m_indices."""
    from dlblas_amd.kernels.fused_moe_v3 import ep_scatter_rows
    print(f'case long row tables T={T} topk={topk} E={E}', flush=True)
    g = helpers.gen(T + E + 1)
    ids = torch.randint(-2, E, (T, topk), generator=g).clamp(min=-1)
    counts = (torch.bincount(ids[ids >= 0], minlength=E) + 127) // 128 * 128
    rows, longer = int(counts.sum()), int(counts.sum()) + 384
    i32 = lambda n, v: torch.full((n, ), v, dtype=torch.int32, device=dev)
    first, m_indices, src, slot = i32(E, -9), i32(longer, -1), i32(longer, 0x7fffffff), torch.full_like(ids, -9, device=dev)
    ep_scatter_rows(ids.to(dev), counts.to(torch.int32).to(dev), first, m_indices, src, slot)
    torch.cuda.synchronize()
    excl, routed, dest = _row_tables_ref(ids, counts)
    src_ref = torch.zeros(longer, dtype=torch.long)
    src_ref[dest[dest >= 0]] = (torch.arange(T * topk) // topk)[dest >= 0]
    assert torch.equal(src.cpu().long(), src_ref)
    assert torch.equal(slot.cpu().flatten(), dest) and torch.equal(first.cpu().long(), excl + routed)
    assert torch.equal(m_indices[:rows].cpu().long(), torch.repeat_interleave(torch.arange(E), counts)) and (m_indices[rows:] == -1).all()


@pytest.mark.parametrize('T,topk,E,dtype,form', [(1, 1, 1, torch.int64, 'whole'), (333, 3, 9, torch.int32, 'whole'), (333, 3, 9, torch.int64, 'whole'),
                                                 (2048, 8, 1, torch.int64, 'whole'), (2047, 8, 77, torch.int32, 'shifted'),
                                                 (1001, 5, 12, torch.int64, 'columns'), (1999, 7, 40, torch.int32, 'transposed'),
                                                 (5000, 1, 6, torch.int64, 'transposed')])
def test_row_tables_from_any_layout_of_ids(dev, T, topk, E, dtype, form):
    """The ids as one array of 16-byte chunks with a remainder, as one that starts off such a boundary, as columns of a
    wider table and column by column; one expert that takes every entry of the largest table ranked in one launch; ids at and past the number of experts."""
    from dlblas_amd.kernels.fused_moe_v3 import ep_scatter_rows
    print(f'case row tables T={T} topk={topk} E={E} {dtype} {form}', flush=True)
    g = helpers.gen(T + E)
    lo, hi = (0, 1) if E == 1 else (-2, E + 2)
    ids = torch.randint(lo, hi, (T, topk), generator=g).to(dtype)
    if form == 'whole':
        on_dev = ids.to(dev)
    elif form == 'shifted':
        on_dev = torch.empty(T * topk + 1, dtype=dtype, device=dev)[1:].view(T, topk).copy_(ids)
    elif form == 'transposed':
        on_dev = torch.empty(topk, T + 1, dtype=dtype, device=dev)[:, :T].t().copy_(ids)
    else:
        on_dev = torch.empty(T, topk + 3, dtype=dtype, device=dev)[:, 1:topk + 1].copy_(ids)
    kept = torch.where(ids < E, ids, -1).clamp(min=-1).long()
    counts = (torch.bincount(kept[kept >= 0], minlength=E) + 127) // 128 * 128
    rows = int(counts.sum())
    i32 = lambda n: torch.full((n, ), -9, dtype=torch.int32, device=dev)
    first, m_indices, src, slot = i32(E), i32(rows), i32(rows), torch.full((T, topk), -9, dtype=torch.int64, device=dev)
    ep_scatter_rows(on_dev, counts.to(torch.int32).to(dev), first, m_indices, src, slot)
    torch.cuda.synchronize()
    excl, routed, dest = _row_tables_ref(kept, counts)
    src_ref = torch.zeros(rows, dtype=torch.long)
    src_ref[dest[dest >= 0]] = (torch.arange(T * topk) // topk)[dest >= 0]
    assert torch.equal(src.cpu().long(), src_ref)
    assert torch.equal(slot.cpu().flatten(), dest) and torch.equal(first.cpu().long(), excl + routed)
    assert torch.equal(m_indices.cpu().long(), torch.repeat_interleave(torch.arange(E), counts))


def test_gathering_gemm_on_a_table_longer_than_the_spans(dev):
    from dlblas_amd.kernels.fp8_gemm_grouped import fp8_gemm_grouped_contiguous_silu_quant
    from dlblas_amd.kernels.fused_moe_v3 import ep_scatter_rows
    print('case gathering GEMM, long row table', flush=True)
    T, topk, E, K, inter = 50, 2, 3, 512, 128
    g = helpers.gen(11)
    x_q, x_s = (t.to(dev) for t in orc.quant_act_1x128(torch.randn(T, K, generator=g).to(torch.bfloat16)))
    ws = [orc.quant_weight_128x128((torch.randn(2 * inter, K, generator=g) * 0.05).to(torch.bfloat16)) for _ in range(E)]
    w_q, w_s = (torch.stack([w[i] for w in ws]).to(dev) for i in (0, 1))
    ids = torch.randint(0, E, (T, topk), generator=g)
    counts = (torch.bincount(ids.flatten(), minlength=E) + 127) // 128 * 128
    rows = int(counts.sum())
    outs = []
    for length in (rows, rows + 256):
        first, slot = torch.empty(E, dtype=torch.int32, device=dev), torch.empty_like(ids, device=dev)
        m_indices = torch.full((length, ), -1, dtype=torch.int32, device=dev)
        src = torch.full((length, ), 0x7fffffff, dtype=torch.int32, device=dev)
        ep_scatter_rows(ids.to(dev), counts.to(torch.int32).to(dev), first, m_indices, src, slot)
        assert int(src.max()) < T  # before the GEMM follows them
        outs.append(fp8_gemm_grouped_contiguous_silu_quant(x_q, x_s, w_q, w_s, m_indices, a_row_index=src))
    torch.cuda.synchronize()
    (q, s), (q2, s2) = outs
    assert torch.equal(q2.view(torch.uint8)[:rows], q.view(torch.uint8)) and torch.equal(s2[:rows], s)


@pytest.mark.parametrize('T,topk,E', [(250, 1, 3), (2300, 8, 40), (5100, 8, 300)])
def test_row_tables_where_more_slots_are_routed_than_reserved(dev, T, topk, E):
    """The slots an expert has no rows for go on into the span behind its own, as ep_scatter lays them: an expert without
    slots of its own follows every one that is too short, so each row has one owner."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fused_moe_v3 import ep_scatter_rows
    print(f'case row tables, short reserve T={T} topk={topk} E={E}', flush=True)
    g = helpers.gen(T + E + 2)
    ids = torch.randint(0, (E + 1) // 2, (T, topk), generator=g) * 2  # even experts only
    ids[ids >= E - 1] = 0  # ... and the last one has none: the rows of all slots are in the table
    routed = torch.bincount(ids.flatten(), minlength=E)
    counts = torch.where(torch.arange(E) % 2 == 0, routed - routed.clamp(max=5), torch.tensor(8))
    counts[-1] += -int(counts.sum()) % 128
    rows = int(counts.sum())
    excl, _, dest = _row_tables_ref(ids, counts)
    src_ref = torch.zeros(rows, dtype=torch.long)
    src_ref[dest] = torch.arange(T * topk) // topk
    i32 = lambda n: torch.full((n, ), -9, dtype=torch.int32, device=dev)
    first, m_indices, src, slot = i32(E), i32(rows), i32(rows), torch.full_like(ids, -9, device=dev)
    ep_scatter_rows(ids.to(dev), counts.to(torch.int32).to(dev), first, m_indices, src, slot)
    torch.cuda.synchronize()
    assert torch.equal(slot.cpu().flatten(), dest) and torch.equal(src.cpu().long(), src_ref)
    start, end = i32(E), i32(E)
    src.fill_(-9)
    if _lib.ep_scatter_rows_host(ids.to(dev), counts.tolist(), start, end, first, m_indices, src, slot):
        held = torch.zeros(rows, dtype=torch.bool)
        held[dest] = True
        got = torch.zeros(rows, dtype=torch.bool)
        for a, b in zip(start.tolist(), end.tolist()):
            got[a:b] = True
        assert torch.equal(got, held) and torch.equal(src.cpu().long(), src_ref)
    else:
        assert E > 256


def _close_codes(q, s, ref_q, ref_s, rows):
    """Sums of K slices are added in another order, 1e-7 of them: a bf16 value next to a rounding boundary moves by its last place,
    and with it at most a code by one step (an eighth of the value, or the smallest code's worth), here and there."""
    got, ref = (x.float() * y.repeat_interleave(128, dim=-1) for x, y in ((q, s), (ref_q, ref_s)))
    got, ref = got[rows], ref[rows]
    step = ref.abs() / 8 + ref_s.repeat_interleave(128, dim=-1)[rows] * 2.0**-9
    assert bool(((got - ref).abs() <= 1.01 * step).all())
    assert float((q.view(torch.uint8)[rows] != ref_q.view(torch.uint8)[rows]).float().mean()) < 1e-2


@pytest.mark.parametrize('masked,M_max,N,K,slices', [
    ([1, 31, 32, 33, 0, 64], 64, 512, 1280, [1, 2, 3]),         # 10 blocks: slices of unequal length, as short as the rings
    ([65, 128, 3], 136, 256, 6784, [1, 5, 8]),                  # 53 blocks: several chunks of the scale table in a slice
    ([i % 4 for i in range(70)], 8, 256, 2304, [2]),            # a second window of 64 experts
])
def test_gate_up_in_two_launches(dev, masked, M_max, N, K, slices):
    """The gate/up projection as partial products of every tile and K slice + one launch that adds, activates and quantises: with
    one slice the bits of the fused kernel, with more what another order of the fp32 sums gives; masked rows keep their content."""
    from dlblas_amd import _lib
    from dlblas_amd.kernels.fp8_gemm_grouped import fp8_gemm_grouped_masked_silu_quant
    a_q, a_s, w_q, w_s, mm = _inputs(masked, M_max, N, K, 70 + N + K, dev)
    G = len(masked)
    rows = torch.arange(M_max, device=dev)[None] < mm[:, None]

    def run(mlp):
        q = torch.full((G, M_max, N // 2), 0x5a, dtype=torch.uint8, device=dev).view(torch.float8_e4m3fn)
        s = torch.full((G, N // 256, M_max), -7.0, device=dev).transpose(1, 2)
        assert fp8_gemm_grouped_masked_silu_quant(a_q, a_s, w_q, w_s, q, s, mm, 0, mlp=mlp)
        torch.cuda.synchronize()
        assert (q.view(torch.uint8)[~rows] == 0x5a).all() and (s[~rows] == -7.0).all()
        return q, s

    _lib.tune('stream', 1)
    ref_q, ref_s = run(False)
    ran = 0
    for i, (knob, shape) in enumerate(zip([2, 3, 4, 5, 6, 8, 9, 10, 11], SHAPES + AHEAD)):
        stages = {256: 4 if i == 0 else 3, 128: 6, 64: 9}[int(shape.split('x')[1].split()[0])]
        for n in slices:
            print(f'case gate/up in two launches masked={masked[:6]} N={N} K={K} {shape} slices={n}', flush=True)
            _lib.tune('stream', knob), _lib.tune('stream_slices', n)
            try:
                plan = _lib.plan_stream_launch(2, M_max, N, K, G, 0, quantising=True, mlp=True)
                if K // 128 // n < stages:  # a slice shorter than the ring: not in this shape
                    assert plan is None
                    continue
                assert plan[3] == n
                q, s = run(True)
            finally:
                _lib.tune('stream', 0), _lib.tune('stream_slices', 0)
            ran += 1
            if n == 1:
                assert torch.equal(q.view(torch.uint8)[rows], ref_q.view(torch.uint8)[rows]) and torch.equal(s[rows], ref_s[rows])
            else:
                _close_codes(q, s, ref_q, ref_s, rows)
    assert ran >= 9


@pytest.mark.parametrize('tokens,E,H,inter', [(30, 8, 2560, 768), (300, 8, 1024, 256), (900, 16, 512, 384), (2500, 4, 768, 128)])
def test_expert_mlps_in_every_form(dev, tokens, E, H, inter):
    """fused_moe_v3 and low_latency_experts from short to long experts, in whichever form their planner picks: native and Python path
    agree, and the result stays within what the quantiser between the GEMMs makes of a last place (the bar of the end-to-end tests)
    of the ring kernels'."""
    from dlblas_amd import _fast, _lib
    from dlblas_amd.kernels.fp8 import per_block_quant_fp8, per_token_group_quant_fp8
    from dlblas_amd.kernels.fused_moe_v3 import fused_moe_v3
    from dlblas_amd.kernels.moe import low_latency_experts
    print(f'case expert MLP forms tokens={tokens} E={E} H={H} I={inter}', flush=True)
    g = helpers.gen(15)

    def weights(n, k):
        q, s = zip(*(per_block_quant_fp8((torch.randn(n, k, generator=g) * 0.05).to(torch.bfloat16).to(dev)) for _ in range(E)))
        return torch.stack(q), torch.stack(s)

    w13, w2 = weights(2 * inter, H), weights(H, inter)
    x = per_token_group_quant_fp8(torch.randn(tokens, H, generator=g).to(torch.bfloat16).to(dev), 128)
    ids = torch.rand(tokens, 4 * E, generator=g).topk(4, dim=1).indices
    ids = torch.where(ids < E, ids, torch.full_like(ids, -1))
    counts = ((torch.bincount(ids[ids >= 0], minlength=E) + 127) // 128 * 128).tolist()
    args = ids.to(dev), torch.rand(tokens, 4, generator=g).to(dev), w13, w2, counts
    valid = torch.bincount(ids[ids >= 0], minlength=E).to(torch.int32)
    cap = int(valid.max()) + 5
    a_q, a_s = per_token_group_quant_fp8(torch.randn(E * cap, H, generator=g).to(torch.bfloat16).to(dev), 128)
    low = (a_q.view(E, cap, H), a_s.view(E, cap, -1)), *w13, *w2, valid.to(dev), max(1, int(valid.float().mean()))
    rows = torch.arange(cap, device=dev)[None] < low[5][:, None]
    outs = []
    for knob in (0, 1):
        _lib.tune('stream', knob)
        out, down = fused_moe_v3(x, *args), low_latency_experts(*low)
        assert _fast.fused_moe_v3(*x, *args[:2], *w13, *w2, counts) is not None
        with torch.overrides.BaseTorchFunctionMode():
            out2, down2 = fused_moe_v3(x, *args), low_latency_experts(*low)
        torch.cuda.synchronize()
        assert torch.equal(out, out2) and torch.equal(down[rows], down2[rows])
        outs.append((out.float(), down[rows].float()))
    _lib.tune('stream', 0)
    for got, ref in zip(*outs):
        assert orc.similarity_gap(got.cpu(), ref.cpu()) <= 1e-4
        assert float((got - ref).abs().max()) <= 0.05 * float(ref.pow(2).mean().sqrt())
