"""GPU parity of the MoE layout helpers (mapping, expansion) against the CPU oracle, bit for bit,
and the end-to-end chain mapping -> expansion -> fused SwiGLU cast.  Structure follows the
reference's tests/moe/test_get_fused_mapping.py and tests/moe/test_expand_to_fused.py."""
import pytest
import torch

from oracle import torch_ref
from tests._util import assert_same
from tests.test_gpu_swiglu import check_fused

pytestmark = pytest.mark.gpu


def _tk():
    import tilekernels_amd
    return tilekernels_amd


def _topk_idx(T, K, E, drop=0.1, seed=0):
    g = torch.Generator().manual_seed(seed)
    scores = torch.rand((T, E), generator=g)
    idx = torch.topk(scores, K, dim=-1).indices
    if drop:
        idx = idx.masked_fill(torch.rand(idx.shape, generator=g) < drop, -1)
    return idx.contiguous()


@pytest.mark.parametrize('alignment', [16, 64, 128])
@pytest.mark.parametrize('T,K,E', [(4001, 8, 256), (4001, 6, 72), (4001, 2, 9), (513, 9, 32), (7, 1, 1), (1, 2, 384), (64, 8, 1024),
                                   (20001, 8, 256), (33000, 4, 9), (16384, 8, 64), (4001, 8, 768)])
def test_get_fused_mapping(T, K, E, alignment):
    tk = _tk()
    topk_idx = _topk_idx(T, K, E, seed=T + K)
    want = torch_ref.get_fused_mapping(topk_idx, E, alignment)
    got = tk.moe.get_fused_mapping(topk_idx.cuda(), E, 0, alignment)
    names = ['pos_to_expert', 'pos_to_token', 'pos_to_token_topk', 'token_topk_to_pos', 'expert_start', 'expert_end', 'num_tokens_per_expert']
    for n, g, w in zip(names, got[:7], want):
        assert_same(g, w, n)
    assert got[7] == want[6].tolist()
    # fixed-size buffer, no host sync: same content, untouched tail marked as padding
    R = want[0].numel() + 3 * alignment
    got2 = tk.moe.get_fused_mapping(topk_idx.cuda(), E, R, alignment)
    assert got2[7] == [] and got2[0].numel() == R
    assert torch.equal(got2[0].cpu()[: want[0].numel()], want[0]) and torch.all(got2[0].cpu()[want[0].numel():] == -1)
    assert_same(got2[3], want[3], 'token_topk_to_pos')


def test_get_fused_mapping_no_tokens():
    tk = _tk()
    got = tk.moe.get_fused_mapping(torch.empty((0, 4), dtype=torch.int64, device='cuda'), 8, 0, 16)
    assert got[0].numel() == 0 and got[7] == [0] * 8 and torch.all(got[4].cpu() == 0)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32, torch.float8_e4m3fn])
@pytest.mark.parametrize('hidden', [128, 576, 2048, 7168])
@pytest.mark.parametrize('T,K,E', [(1001, 8, 64), (257, 2, 9), (3, 1, 4), (9, 3, 5)])
def test_expand_to_fused(T, K, E, hidden, dtype):
    tk = _tk()
    topk_idx = _topk_idx(T, K, E, seed=hidden)
    p2e, _, _, t2p, *_ = torch_ref.get_fused_mapping(topk_idx, E, 16)
    x = torch.randn((T, hidden)).to(dtype)
    want = torch_ref.expand_to_fused(x, t2p, p2e)
    got = tk.moe.expand_to_fused(x.cuda(), t2p.cuda(), p2e.cuda())
    assert_same(got, want, 'expanded')


@pytest.mark.parametrize('mode', [(False, True, False), (True, True, True), (True, False, False), (False, False, False)],
                         ids=lambda m: 'col%d-round%d-packed%d' % tuple(int(v) for v in m))
@pytest.mark.parametrize('num_per_channels', [32, 128])
@pytest.mark.parametrize('hidden', [576, 4096])
def test_expand_to_fused_with_sf(hidden, num_per_channels, mode):
    tk = _tk()
    col, rnd, packed = mode
    T, K, E = 777, 6, 72
    topk_idx = _topk_idx(T, K, E, seed=hidden + num_per_channels)
    p2e, _, _, t2p, *_ = torch_ref.get_fused_mapping(topk_idx, E, 16)
    x = torch.randn((T, hidden)).to(torch.bfloat16)
    codes, sf = torch_ref.cast(x, 'e4m3', (1, num_per_channels), round_sf=rnd, use_tma_aligned_col_major_sf=col, use_packed_ue8m0=packed)
    sf = torch.empty(sf.shape, dtype=sf.dtype).copy_(sf)
    want = torch_ref.expand_to_fused_with_sf((codes, sf), num_per_channels, t2p, p2e, col)
    got = tk.moe.expand_to_fused_with_sf((codes.cuda(), sf.cuda()), num_per_channels, t2p.cuda(), p2e.cuda(), col)
    assert_same(got[0], want[0], 'codes')
    assert_same(got[1], want[1], 'sf')


def test_moe_chain_mapping_expand_swiglu_cast():
    """The three steps as an MoE layer runs them, all on the GPU, against the same chain on the CPU."""
    tk = _tk()
    T, K, E, H = 1024, 8, 64, 1024
    g = torch.Generator().manual_seed(3)
    logits = torch.randn((T, E), generator=g)
    w, idx = torch.topk(torch.softmax(logits, -1), K, dim=-1)
    x = torch.randn((T, 2 * H), generator=g).to(torch.bfloat16)
    p2e, _, p2tk, t2p, *_ = torch_ref.get_fused_mapping(idx, E, 128)
    want = torch_ref.swiglu_forward_and_per_token_cast(torch_ref.expand_to_fused(x, t2p, p2e), 'e4m3', 128, p2tk, w.contiguous(), p2e)
    m = tk.moe.get_fused_mapping(idx.cuda().contiguous(), E, 0, 128)
    xe = tk.moe.expand_to_fused(x.cuda(), m[3], m[0])
    got = tk.quant.swiglu_forward_and_per_token_cast(xe, 'e4m3', 128, m[2], w.cuda().contiguous(), m[0])
    check_fused(got, want, H // 128, False, 'chain')


@pytest.mark.parametrize('K', [1, 8, 11, 70])
@pytest.mark.parametrize('T,dim,dtype', [(37, 16, torch.bfloat16), (37, 1024, torch.bfloat16), (37, 1032, torch.bfloat16), (9, 2048, torch.float8_e4m3fn),
                                         (9, 7168, torch.float8_e4m3fn), (33, 4096, torch.bfloat16)])
@pytest.mark.parametrize('live', [0.0, 0.15, 1.0])
def test_expand_to_fused_sparse_and_full_lists(T, K, dim, dtype, live):
    """One workgroup per token: lists with no, few and all positions set, beyond one ballot, rows shorter than, equal to and
    longer than a chunk (4 KB)."""
    tk = _tk()
    g = torch.Generator().manual_seed(T * K + dim)
    here = torch.rand((T, K), generator=g) < live
    R = int(here.sum()) + 5
    t2p = torch.full((T, K), -1, dtype=torch.int32)
    t2p[here] = torch.randperm(R, generator=g)[:int(here.sum())].to(torch.int32)
    p2e = torch.full((R,), -1, dtype=torch.int32)
    p2e[t2p[here].long()] = 3
    x = torch.randn((T, dim), generator=g).to(dtype)
    want = torch_ref.expand_to_fused(x.view(torch.uint8), t2p, p2e)
    got = tk.moe.expand_to_fused(x.cuda(), t2p.cuda(), p2e.cuda())
    assert torch.equal(got.cpu().view(torch.uint8), want)


@pytest.mark.parametrize('dim', [512, 8192])
def test_expand_to_fused_long_output_with_full_lists(dim):
    """Outputs beyond 160 MB with several positions per token take a workgroup per list entry."""
    tk = _tk()
    T, K = (170 << 20) // (dim * 2) // 4, 4
    g = torch.Generator().manual_seed(dim)
    t2p = torch.randperm(T * K, generator=g).to(torch.int32).view(T, K)
    t2p[::7, 1] = -1
    p2e = torch.full((T * K,), -1, dtype=torch.int32)
    p2e[t2p[t2p >= 0].long()] = 0
    x = torch.randn((T, dim), generator=g).to(torch.bfloat16).cuda()
    got = tk.moe.expand_to_fused(x, t2p.cuda(), p2e.cuda())
    assert T * K * dim * 2 >= 160 << 20
    want = torch.zeros_like(got)
    for k in range(K):
        here = (t2p[:, k] >= 0).cuda()
        want[t2p[:, k].cuda()[here].long()] = x[here]
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize('T,K,E,drop,alignment', [(65536, 1, 1, 0.0, 128), (65537, 1, 512, 0.0, 16), (8200, 8, 3, 0.9, 128), (12000, 6, 9, 1.0, 16),
                                                  (95000, 8, 256, 0.9, 128), (100001, 9, 4, 0.5, 64), (230400, 8, 1, 0.3, 128), (230401, 8, 1, 0.3, 16)])
def test_mapping_of_long_lists(T, K, E, drop, alignment):
    """Lists from 64 Ki pairs on, which are counted into a table first (95000 x 8 of 256 experts, and
    230401 x 8 of one: too long for it, three launches);
    buffers that are longer, and shorter, than the expanded rows."""
    tk = _tk()
    g = torch.Generator().manual_seed(T)
    idx = torch.randint(0, E, (T, K), generator=g)
    idx = idx.masked_fill(torch.rand(idx.shape, generator=g) < drop, -1).contiguous()
    want = torch_ref.get_fused_mapping(idx, E, alignment)
    rows = want[0].numel()
    for extra in (0, 1000, -(rows // 3)):
        got = tk.moe.get_fused_mapping(idx.cuda(), E, rows + extra, alignment, force_no_sync=True)
        n = min(rows, rows + extra)
        for name, a, b in zip(('pos_to_expert', 'pos_to_token', 'pos_to_token_topk'), got[:3], want[:3]):
            assert torch.equal(a.cpu()[:n], b[:n]) and bool((a.cpu()[n:] == -1).all()), (name, extra)
        for a, b, name in zip(got[3:7], want[3:7], ('token_topk_to_pos', 'expert_start', 'expert_end', 'num_tokens_per_expert')):
            assert_same(a, b, name)


@pytest.mark.parametrize('col_major', [False, True], ids=['row', 'col'])
@pytest.mark.parametrize('live', [0.2, 1.0])
@pytest.mark.parametrize('T,K,row_bytes,sf_cols,pad', [(9, 8, 4096, 32, 40), (63, 8, 4096, 32, 300), (64, 4, 4096, 300, 300), (70, 3, 9216, 288, 9),
                                                       (127, 8, 2048, 16, 600), (129, 8, 2048, 200, 600), (300, 2, 1024, 100, 500), (33, 70, 1040, 65, 0)])
def test_expand_to_fused_scale_words(T, K, row_bytes, sf_cols, pad, live, col_major):
    """A workgroup per list entry (few tokens) and per token, with fewer and with more scale words than threads per row."""
    from tilekernels_amd import _ffi
    g = torch.Generator().manual_seed(T * K + sf_cols)
    here = torch.rand((T, K), generator=g) < live
    n = int(here.sum())
    R = n + pad
    t2p = torch.full((T, K), -1, dtype=torch.int32)
    t2p[here] = torch.randperm(R, generator=g)[:n].to(torch.int32)
    p2e = torch.full((R,), -1, dtype=torch.int32)
    p2e[t2p[here].long()] = 1
    x = torch.randint(0, 256, (T, row_bytes), generator=g, dtype=torch.uint8)
    sf = torch.randint(-2 ** 31, 2 ** 31 - 1, (T, sf_cols), generator=g, dtype=torch.int32)
    want, want_sf = torch.zeros((R, row_bytes), dtype=torch.uint8), torch.zeros((R, sf_cols), dtype=torch.int32)
    token = torch.arange(T)[:, None].expand(T, K)[here]
    want[t2p[here].long()], want_sf[t2p[here].long()] = x[token], sf[token]
    xg, sg, tg, pg = x.cuda(), sf.cuda(), t2p.cuda(), p2e.cuda()
    out = torch.full((R, row_bytes), 0x5A, dtype=torch.uint8, device='cuda')
    ld = R + 3 if col_major else sf_cols + 3
    out_sf = torch.full((sf_cols if col_major else R, ld), 0x5A5A5A5A, dtype=torch.int32, device='cuda')
    rc = _ffi.load().tk_expand_to_fused(xg.data_ptr(), T, row_bytes, tg.data_ptr(), K, pg.data_ptr(), R, out.data_ptr(), sg.data_ptr(), sf_cols,
                                        out_sf.data_ptr(), ld, int(col_major), torch.cuda.current_stream().cuda_stream)
    assert rc == 0, rc
    assert torch.equal(out.cpu(), want)
    got = out_sf.cpu()
    assert bool((got[:, -3:] == 0x5A5A5A5A).all())
    assert torch.equal(got[:, :-3].T.contiguous() if col_major else got[:, :-3], want_sf)


@pytest.mark.parametrize('T,K,E', [(1, 1, 1), (2, 1, 3), (3, 1, 2), (1, 4, 4), (5, 3, 8), (1365, 3, 32), (4097, 4, 64), (5462, 3, 72),      # one workgroup per expert
                                   (65537, 1, 512), (16500, 4, 9), (230401, 8, 1)])                                                   # a table; three launches
def test_mapping_of_a_list_between_16_byte_boundaries(T, K, E):
    """A contiguous list that starts 8 bytes off (a slice of a longer one): the kernels read pairs from the boundary on, and the first
    (and, of an even number, the last) entry by itself."""
    tk = _tk()
    g = torch.Generator().manual_seed(T + K)
    idx = torch.randint(-1, E, (T, K), generator=g)
    idx[0, 0] = idx[-1, -1] = E - 1
    want = torch_ref.get_fused_mapping(idx, E, 16)
    buf = torch.empty((T * K + 1,), dtype=torch.int64, device='cuda')
    buf[0] = 0                      # an entry in front of the list that would count
    view = buf[1:].view(T, K)
    view.copy_(idx)
    assert view.data_ptr() % 16 == 8 and view.is_contiguous()
    for got in (tk.moe.get_fused_mapping(view, E, 0, 16), tk.moe.get_fused_mapping(view, E, want[0].numel(), 16)):
        for name, a, b in zip(('pos_to_expert', 'pos_to_token', 'pos_to_token_topk', 'token_topk_to_pos', 'expert_start', 'expert_end',
                               'num_tokens_per_expert'), got[:7], want):
            assert_same(a, b, name)


@pytest.mark.parametrize('T,K,E,alignment', [(57, 9, 256, 128), (1, 1, 512, 128), (300, 8, 512, 128), (3, 2, 64, 1024)])
def test_mapping_of_short_lists_into_long_buffers(T, K, E, alignment):
    """More workgroups than the list has pairs for: they mark the padding of experts and of the buffer's end."""
    tk = _tk()
    g = torch.Generator().manual_seed(T * E)
    idx = torch.randint(-1, E, (T, K), generator=g)
    want = torch_ref.get_fused_mapping(idx, E, alignment)
    rows = want[0].numel()
    got = tk.moe.get_fused_mapping(idx.cuda(), E, 0, alignment)
    for a, b in zip(got[:7], want[:7]):
        assert torch.equal(a.cpu(), b)
    for extra in (1, 70_001):
        got = tk.moe.get_fused_mapping(idx.cuda(), E, rows + extra, alignment)
        for a, b in zip(got[:3], want[:3]):
            assert torch.equal(a[:rows].cpu(), b) and bool((a[rows:] == -1).all())
        for a, b in zip(got[3:7], want[3:7]):
            assert torch.equal(a.cpu(), b)


# one launch, two around a table, three; behind an idle stream and behind work that takes longer than the wait in a loop
@pytest.mark.parametrize('busy', [False, True])
@pytest.mark.parametrize('T,K,E', [(1, 1, 1), (700, 6, 512), (11000, 8, 32), (90, 5, 700), (0, 4, 8)])
def test_segment_lengths_on_the_host(T, K, E, busy):
    from tilekernels_amd import _ffi
    tk = _tk()
    g = torch.Generator().manual_seed(T + E)
    idx = torch.randint(-1, E, (T, K), generator=g)
    want = torch_ref.get_fused_mapping(idx, E, 16) if T else None
    idx = idx.cuda()
    if busy:
        torch.cuda._sleep(5_000_000)
    got = tk.moe.get_fused_mapping(idx, E, 0, 16)
    assert got[7] == got[6].tolist() and got[0].shape[0] == sum(got[7])
    if T == 0:
        return
    for a, b in zip(got[:7], want[:7]):
        assert torch.equal(a.cpu(), b)
    lib, i32 = _ffi.load(), dict(dtype=torch.int32, device='cuda')
    rows = (T * K + 15 * E) // 16 * 16
    out = [torch.empty((max(rows, T * K, E),), **i32) for _ in range(7)]
    ws = torch.empty((lib.tk_fused_mapping_workspace_bytes(T, K, E) // 4,), **i32)
    host = torch.empty((E,), dtype=torch.int32, pin_memory=True)

    def call(counts, stream):
        return lib.tk_get_fused_mapping_with_counts(idx.data_ptr(), T, K, E, 16, rows, *(t.data_ptr() for t in out), ws.data_ptr(), ws.numel() * 4,
                                                    counts, stream)
    if busy:
        torch.cuda._sleep(5_000_000)
    assert call(host.data_ptr(), _ffi.current_stream(idx.device)) == 0
    assert host.tolist() == got[7]
    assert call(None, _ffi.current_stream(idx.device)) == -1                    # null pointer
    assert call(torch.empty((E,), dtype=torch.int32).data_ptr(), _ffi.current_stream(idx.device)) == -11        # memory the GPU cannot write
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        rc = call(host.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == -7                                                             # nothing runs during a capture: no lengths to wait for


# one launch, two around a table, three
@pytest.mark.parametrize('T,K,E', [(700, 6, 512), (50_000, 8, 32), (400_000, 8, 700)])
def test_a_trimming_call_returns_when_the_stream_is_through(T, K, E):
    """As behind a copy of the lengths to the host, the lists may be read on another stream without an event."""
    tk = _tk()
    idx = torch.randint(-1, E, (T, K), generator=torch.Generator().manual_seed(T)).cuda()
    want = tk.moe.get_fused_mapping(idx, E, (T * K + 15 * E) // 16 * 16, 16)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for _ in range(3):
        got = tk.moe.get_fused_mapping(idx, E, 0, 16)
        assert torch.cuda.current_stream().query()
        with torch.cuda.stream(side):
            there = [t.clone() for t in got[:7]]
        torch.cuda.synchronize()
        for a, b in zip(there, want[:7]):
            assert torch.equal(a, b[:len(a)])
