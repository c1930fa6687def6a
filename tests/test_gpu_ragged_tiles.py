"""Casts whose last tile overhangs the matrix, bit for bit against the oracle: fp32 rows that end inside a run of lanes (the run's
loads are dealt out through LDS), per-block tiles at the lower and right edge (lanes beyond it read the last row or column
instead), and the two tile widths of the per-channel cast on either side of the line between them."""
import pytest
import torch

from oracle import torch_ref
from tests._util import assert_same

pytestmark = pytest.mark.gpu

LAYOUTS = {'row': {}, 'col': dict(use_tma_aligned_col_major_sf=True),
           'packed': dict(use_tma_aligned_col_major_sf=True, round_sf=True, use_packed_ue8m0=True)}


def _matrix(M, K, dtype):
    x = torch.randn((M, K), generator=torch.Generator().manual_seed(M * 7 + K))
    x[-1] *= 100          # the last row and the last columns decide the scales of their blocks
    x[:, -8:] *= 30
    x[:, 0] *= 1000       # (and would show in other blocks if lanes beyond the edge read the first ones)
    return x.to(dtype)


@pytest.mark.parametrize('layout', LAYOUTS)
@pytest.mark.parametrize('fmt,group', [('e4m3', 128), ('e4m3', 16), ('e2m1', 32)])
@pytest.mark.parametrize('M,K', [(1, 1024), (9, 1536), (7, 1544), (130, 2824), (33, 264), (5, 136), (66, 72), (257, 2560)])
def test_per_token_fp32(M, K, fmt, group, layout):
    import tilekernels_amd as tk
    x = _matrix(M, K, torch.float32)
    got, want = tk.quant.per_token_cast(x.cuda(), fmt, group, **LAYOUTS[layout]), torch_ref.cast(x, fmt, (1, group), **LAYOUTS[layout])
    assert_same(got[0], want[0], 'codes')
    assert_same(got[1], want[1], 'scales')


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
@pytest.mark.parametrize('block', [(128, 128), (32, 32), (128, 32)])
@pytest.mark.parametrize('M,K', [(1, 64), (127, 192), (129, 320), (300, 576), (4001, 2112), (3999, 2048)])
def test_per_block_edges(M, K, block, dtype):
    import tilekernels_amd as tk
    x = _matrix(M, K, dtype)
    got, want = tk.quant.per_block_cast(x.cuda(), 'e4m3', block), torch_ref.cast(x, 'e4m3', block)
    assert_same(got[0], want[0], 'codes')
    assert_same(got[1], want[1], 'scales')


@pytest.mark.parametrize('num_per_tokens', [32, 128])
@pytest.mark.parametrize('M,K', [(128, 64), (256, 192), (1920, 4096), (2048, 4096), (2176, 4096), (2048, 4160)])      # 1, 2, 240, 256, 272, 272 tiles of 256 columns: narrow below 256
def test_per_channel_transposed(M, K, num_per_tokens):
    import tilekernels_amd as tk
    x = _matrix(M, K, torch.bfloat16)
    got = tk.quant.per_channel_cast_and_transpose(x.cuda(), 'e4m3', num_per_tokens)
    want = torch_ref.per_channel_cast_and_transpose(x, num_per_tokens, False)
    assert_same(got[0], want[0], 'codes')
    assert_same(got[1], want[1], 'scales')


@pytest.mark.parametrize('M,K', [(16, 128), (144, 640), (1920, 8192), (2048, 8192)])                      # 1, 4, 240, 256 tiles of 512 columns
def test_per_channel_gathered_codes(M, K):
    import tilekernels_amd as tk
    g = torch.Generator().manual_seed(M)
    T = max(M // 2, 3)
    codes = torch_ref.cast(_matrix(T, K, torch.bfloat16), 'e4m3', (1, 128))
    pos = torch.randint(-1, T, (M,), generator=g, dtype=torch.int32)
    got = tk.quant.per_channel_cast_fused((codes[0].cuda(), codes[1].cuda()), 'e4m3', 128, num_per_channels=128, pos_to_token=pos.cuda())
    want = torch_ref.per_channel_cast_fused(codes, 128, 128, False, pos)
    assert_same(got[0], want[0], 'codes')
    assert_same(got[1], want[1], 'scales')


@pytest.mark.parametrize('kind,transpose,gather', [('bf16', False, False), ('bf16', False, True), ('bf16', True, False), ('bf16', True, True),
                                                   ('fp32', False, False), ('fp32', False, True), ('e4m3', False, False), ('e4m3', False, True),
                                                   ('e4m3', True, False), ('e4m3', True, True), ('swiglu', False, False), ('swiglu', True, False)])
@pytest.mark.parametrize('num_per_tokens', [32, 128])
def test_per_channel_tile_widths_agree(kind, transpose, gather, num_per_tokens):
    """One call on a matrix that takes wide tiles against calls on its pieces of 512 rows, which take narrow ones (no scale spans two
    pieces): every form of tk_per_channel_cast, also those the Python functions do not ask for and codes aligned to 8 bytes."""
    from tilekernels_amd import _ffi
    lib = _ffi.load()
    M, K = 2176, 8320 if kind == 'e4m3' and not transpose else 4224                # 289 wide tiles; 68 and fewer in a piece
    g = torch.Generator(device='cuda').manual_seed(K)
    width = 2 * K if kind == 'swiglu' else K
    x = torch.randn((M, width), generator=g, device='cuda')
    x = x if kind == 'fp32' else x.to(torch.bfloat16)
    sf = None
    if kind == 'e4m3':
        x, sf = x.to(torch.float8_e4m3fn), torch.rand((M, K // 128), generator=g, device='cuda') + 0.1
    pos = torch.randint(-1, M, (M,), generator=g, device='cuda', dtype=torch.int32) if gather else None
    x = x.view(torch.uint8)

    def cast(first, rows, shift):
        lo = 0 if gather else first
        data = torch.zeros((M - lo) * x.shape[1] + 16, dtype=torch.uint8, device='cuda')
        data[shift:shift + (M - lo) * x.shape[1]] = x[lo:].reshape(-1)
        out = torch.zeros(rows * K + 16, dtype=torch.uint8, device='cuda')
        out_sf = torch.zeros((-(-rows // num_per_tokens), K), device='cuda')
        sub_sf, sub_pos = None if sf is None else sf[lo:], None if pos is None else pos[first:]
        rc = lib.tk_per_channel_cast(data.data_ptr() + shift, int(kind == 'fp32'), _ffi.ptr(sub_sf), M - lo, K, _ffi.ptr(sub_pos), rows,
                                     out.data_ptr() + shift, out_sf.data_ptr(), num_per_tokens, 1, int(transpose), int(kind == 'swiglu'),
                                     int(kind == 'swiglu'), 1.5 if kind == 'swiglu' else 0.0, _ffi.current_stream(x.device))
        assert rc == 0, rc
        out = out[shift:shift + rows * K]
        return (out.view(K, rows).T if transpose else out.view(rows, K)), out_sf

    for shift in (0, 8) if kind == 'e4m3' and not transpose else (0,):
        codes, scales = cast(0, M, shift)
        pieces = [cast(first, min(512, M - first), shift) for first in range(0, M, 512)]
        assert torch.equal(codes, torch.cat([p[0] for p in pieces])) and torch.equal(scales, torch.cat([p[1] for p in pieces]))


@pytest.mark.parametrize('clamp', [None, 1.5])
@pytest.mark.parametrize('weighted', [False, True])
@pytest.mark.parametrize('R,H', [(6145, 2048), (8190, 2048), (8191, 2048), (4099, 4096), (2051, 8192), (8189, 2560), (6545, 2560), (10921, 1536), (2049, 7168),
                                 (32771, 512)])
def test_swiglu_launches_that_end_in_smaller_waves_on_any_row_count(R, H, weighted, clamp):
    """Row-major scales, rows that are no multiple of the tiles (H a multiple of 2048: row-wise tiles, else stacked): one call against calls on pieces of 999 rows, which are too small to end in
    smaller waves."""
    import tilekernels_amd as tk
    g = torch.Generator(device='cuda').manual_seed(R)
    x = (torch.randn((R, 2 * H), generator=g, device='cuda') * 2).to(torch.bfloat16)
    slots = torch.randint(-1, R, (R,), generator=g, device='cuda', dtype=torch.int32) if weighted else None
    weights = torch.rand((R, 1), generator=g, device='cuda') if weighted else None
    op = tk.quant.swiglu_forward_and_per_token_cast
    codes, sf = op(x, 'e4m3', 128, slots, weights, swiglu_clamp_value=clamp)
    pieces = [op(x[i:i + 999], 'e4m3', 128, None if slots is None else slots[i:i + 999], weights, swiglu_clamp_value=clamp) for i in range(0, R, 999)]
    assert torch.equal(codes.view(torch.uint8), torch.cat([p[0].view(torch.uint8) for p in pieces]))
    assert torch.equal(sf, torch.cat([p[1] for p in pieces]))


# fp32 tiles that overhang the matrix: launches of fewer than 256 workgroups load each lane's elements directly, larger ones deal whole-line
# loads out between the lanes.  4101 rows of each length here are more than that and 499 rows fewer, in the tiles they take.
FEW, MANY = 499, 4101


def _both_sides(cast, x):
    whole = cast(x)
    pieces = [cast(x[i:i + FEW]) for i in range(0, MANY, FEW)]
    for i, part in enumerate(whole):
        assert torch.equal(part.contiguous().view(torch.uint8), torch.cat([p[i] for p in pieces]).contiguous().view(torch.uint8)), f'output {i}'
    return pieces[-1], x[MANY // FEW * FEW:]


@pytest.mark.parametrize('group', [16, 32, 64, 128])
@pytest.mark.parametrize('fmt', ['e4m3', 'e2m1'])
@pytest.mark.parametrize('K', [512, 896, 1408, 1536, 320, 640])       # one strip, two, three (one wide tile; ragged, whole), short rows end to end
def test_per_token_fp32_few_and_many_workgroups(K, fmt, group):
    import tilekernels_amd as tk
    if K % group:
        pytest.skip('rows are whole groups')
    x = _matrix(MANY, K, torch.float32).cuda()
    last, rows = _both_sides(lambda v: tk.quant.per_token_cast(v, fmt, group), x)
    want = torch_ref.cast(rows.cpu(), fmt, (1, group))
    assert_same(last[0], want[0], 'codes')
    assert_same(last[1], want[1], 'scales')
    _both_sides(lambda v: (tk.quant.per_token_cast_with_sf_only(v, fmt, group),), x)
    sf = torch.rand((1, K // group), device='cuda') + 0.5
    _both_sides(lambda v: (tk.quant.per_token_cast_with_precomputed_sf(v, fmt, group, sf.repeat(v.shape[0], 1)),), x)
    assert_same(tk.quant.per_token_cast_with_sf_only(rows, fmt, group), want[1], 'scales alone')


@pytest.mark.parametrize('with_mask', [False, True])
@pytest.mark.parametrize('mode', ['plain', 'clamp', 'count'])
@pytest.mark.parametrize('H,layout', [(512, 'row'), (896, 'row'), (2560, 'row'), (640, 'row'), (1024, 'col'), (2048, 'packed')])
def test_swiglu_fp32_few_and_many_workgroups(H, layout, mode, with_mask):
    import tilekernels_amd as tk
    from tests.test_gpu_swiglu import check_fused
    g = torch.Generator().manual_seed(H)
    x = torch.randn((MANY, 2 * H), generator=g) * 2
    pe = torch.randint(-1, 4, (MANY,), generator=g, dtype=torch.int32)
    clamp = None if mode == 'plain' else 1.0

    def run(v, first, rows):
        count = torch.zeros(3, dtype=torch.int64, device=v.device) if mode == 'count' else None
        kw = dict(swiglu_clamp_value=clamp, clamped_count=count, **LAYOUTS[layout])
        m = pe[first:first + rows].to(v.device) if with_mask else None
        return (tk.quant if v.is_cuda else torch_ref).swiglu_forward_and_per_token_cast(v[first:first + rows], 'e4m3', 128, pos_to_expert=m, **kw), count

    xd = x.cuda()
    (codes, sf), count = run(xd, 0, MANY)
    pieces = [run(xd, i, FEW) for i in range(0, MANY, FEW)]
    assert torch.equal(codes.view(torch.uint8), torch.cat([p[0][0].view(torch.uint8) for p in pieces]))
    assert torch.equal(sf, torch.cat([p[0][1] for p in pieces]))
    if count is not None:
        assert torch.equal(count, sum(p[1] for p in pieces)) and count.sum() > 0
    first = MANY // FEW * FEW
    check_fused(pieces[-1][0], run(x, first, FEW)[0], H // 128, layout == 'packed')


@pytest.mark.parametrize('fmt', ['e4m3', 'e2m1'])
@pytest.mark.parametrize('block', [(128, 128), (32, 32), (128, 32), (32, 128)])
@pytest.mark.parametrize('M', [1, 31, 32, 63, 64, 65])
def test_per_block_fp32_few_rows(M, block, fmt):
    import tilekernels_amd as tk
    for K in (64, 192, 2560):
        x = _matrix(M, K, torch.float32)
        got, want = tk.quant.per_block_cast(x.cuda(), fmt, block), torch_ref.cast(x, fmt, block)
        assert_same(got[0], want[0], 'codes')
        assert_same(got[1], want[1], 'scales')
