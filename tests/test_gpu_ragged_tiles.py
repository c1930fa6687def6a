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
