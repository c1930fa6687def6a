"""The native call path of the ops against their Python code: the same results in the same layout for every form both accept,
and None (so that the Python code takes the call) for the forms it leaves alone."""
import itertools
import os

import pytest
import torch


class Recorder:
    """Stands in for the native functions: counts the calls they took, or leaves all of them to the Python code."""

    def __init__(self, native):
        self.native, self.taken = native, 0

    def __getattr__(self, name):
        def call(*args):
            if self.native is None:
                return None
            r = getattr(self.native, name)(*args)
            self.taken += r is not None
            return r
        return call


def _flat(r):
    return [v for item in r for v in _flat(item)] if isinstance(r, (tuple, list)) else [r]


def _bytes(t):
    return t.cpu().clone(memory_format=torch.contiguous_format).view(-1).view(torch.uint8)


def _compare(monkeypatch, calls, native=True):
    from tilekernels_amd import _ffi
    _ffi.host.per_token_cast        # load
    host = _ffi.host
    for name, call in calls:
        recorder = Recorder(host)
        monkeypatch.setattr(_ffi, 'host', recorder)
        got = call()
        assert bool(recorder.taken) == native, (name, recorder.taken)
        monkeypatch.setattr(_ffi, 'host', Recorder(None))
        want = call()
        monkeypatch.setattr(_ffi, 'host', host)
        for g, w in zip(_flat(got), _flat(want), strict=True):
            if isinstance(w, int):
                assert g == w, name
                continue
            assert (g.dtype, g.shape, g.stride(), g.device, g.requires_grad) == (w.dtype, w.shape, w.stride(), w.device, w.requires_grad), name
            assert g.untyped_storage().nbytes() == w.untyped_storage().nbytes(), name
            assert torch.equal(_bytes(g), _bytes(w)), name


LAYOUTS = [(False, False, False), (False, True, False), (True, False, False), (True, True, True)]


def _x(rows, cols, dtype=torch.bfloat16, scale=1.0):
    g = torch.Generator().manual_seed(rows * 131 + cols)
    return (torch.randn((rows, cols), generator=g) * scale).to(dtype).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize('rows', [1, 3, 65])
def test_casts_and_dequantisation(monkeypatch, rows):
    import tilekernels_amd as tk
    q, calls = tk.quant, []
    for dtype, layout in itertools.product((torch.bfloat16, torch.float32), LAYOUTS):
        for cols, fmt, group in ((512, 'e4m3', 128), (576, 'e4m3', 64), (704, 'e2m1', 32), (64, 'e4m3', 16), (576, 'e4m3', 576), (584, 'e5m6', 584)):
            x = _x(rows, cols, dtype)
            calls.append(((dtype, layout, cols, fmt), lambda x=x, f=fmt, g=group, l=layout: q.per_token_cast(x, f, g, None, *l)))
            wide = _x(rows, cols + 64, dtype)[:, :cols]
            calls.append(((dtype, layout, cols, fmt, 'strided'), lambda x=wide, f=fmt, g=group, l=layout: q.per_token_cast(x, f, g, None, *l)))
        for fmt, block in (('e4m3', (128, 128)), ('e2m1', (32, 32)), ('e4m3', (32, 128))):
            x = _x(rows, 320, dtype)
            calls.append(((dtype, layout, fmt, block), lambda x=x, f=fmt, b=block, l=layout: q.per_block_cast(x, f, b, *l)))
    for fmt, group, layout in (('e4m3', 128, LAYOUTS[0]), ('e4m3', 32, LAYOUTS[2]), ('e2m1', 32, LAYOUTS[3]), ('e4m3', 64, LAYOUTS[3]),
                               ('e2m1', 128, LAYOUTS[0])):
        for cols in (128, 1088):
            codes = q.per_token_cast_with_sf_only(_x(rows, cols), fmt, group, None, *layout), q.per_token_cast(_x(rows, cols), fmt, group, None, *layout)
            codes = (codes[1][0], codes[0])
            for back in ('bf16', 'fp32'):
                calls.append(((fmt, group, layout, cols, back), lambda c=codes, b=back, g=group: q.per_token_cast_back(c, b, g)))
            for out in LAYOUTS:
                calls.append(((fmt, group, layout, cols, out), lambda c=codes, g=group, l=out: q.per_token_cast(c, 'e4m3', 32, (1, g), *l)))
    codes = q.per_token_cast(_x(rows, 584), 'e5m6', 584)
    calls.append(('e5m6', lambda: q.per_token_cast_back(codes, 'bf16', 584, 'e5m6')))
    _compare(monkeypatch, calls)


@pytest.mark.gpu
@pytest.mark.parametrize('tokens,hidden', [(1, 256), (97, 768)])
def test_expanded_ops(monkeypatch, tokens, hidden):
    import tilekernels_amd as tk
    q, moe, calls = tk.quant, tk.moe, []
    g = torch.Generator().manual_seed(tokens)
    idx = torch.topk(torch.rand((tokens, 16), generator=g), 4, dim=-1).indices
    idx = idx.masked_fill(idx > 7, -1)
    idx[0, 0] = 3
    idx, weights = idx.cuda(), torch.rand((tokens, 4), generator=g).cuda()
    for args in ((8, 0, 16), (8, 0, 64), (8, 2048, 16), (8, 0, 16, True)):
        def mapping(args=args):
            m = moe.get_fused_mapping(idx, *args)
            return m if args[1] == 0 and len(args) == 3 else (m[3:7], m[7])     # (buffers longer than the live rows have an unwritten end)
        calls.append((args, mapping))
    maps = moe.get_fused_mapping(idx, 8, 0, 16)
    p2e, p2t, p2tk, t2p = maps[:4]
    rows = p2e.shape[0]
    x = _x(tokens, hidden)
    calls.append(('expand', lambda: moe.expand_to_fused(x, t2p, p2e)))
    for layout in (LAYOUTS[0], LAYOUTS[3]):
        codes, sf = q.per_token_cast(x, 'e4m3', 128, None, *layout)
        for col in ((True,) if sf.dtype == torch.int32 else (False, True)):
            calls.append((('expand', layout, col), lambda c=codes, s=sf.contiguous(), col=col: moe.expand_to_fused_with_sf((c, s), 128, t2p, p2e, col)))
    y = _x(rows, hidden)
    row_sf, one = torch.rand((rows,), generator=g).cuda(), torch.full((1,), 0.5, device='cuda')
    for dtype in (torch.bfloat16, torch.float32):
        for args in ((y.to(dtype), None, t2p), (y.to(dtype), weights, t2p), ((y.to(dtype), row_sf), weights, t2p), (y.to(dtype), weights, t2p, 'e4m3', one)):
            calls.append((('reduce', dtype, len(args)), lambda args=args: moe.reduce_fused(*args)))
        z = _x(rows, 2 * hidden, dtype, 2.0)
        for layout, clamp in itertools.product(LAYOUTS, (None, 1.5)):
            calls.append((('swiglu', dtype, layout, clamp),
                          lambda z=z, l=layout, c=clamp: q.swiglu_forward_and_per_token_cast(z, 'e4m3', 128, p2tk, weights, p2e, *l, swiglu_clamp_value=c)))
        calls.append((('swiglu row', dtype), lambda z=z: q.swiglu_forward_and_per_token_cast(z, 'e4m3', hidden, sf_clamp_min=1e-3)))
    for group, clamp in ((32, None), (128, 1.5)):
        codes = q.per_token_cast(_x(rows, 2 * hidden, scale=2.0), 'e4m3', group)
        calls.append((('backward', group), lambda c=codes, g=group, cl=clamp: q.swiglu_backward_and_per_token_cast(c, y, weights, p2tk, t2p, g,
                                                                                                                   swiglu_clamp_value=cl)))
    t = _x(128, hidden)
    quantised = q.per_token_cast(_x(tokens, hidden), 'e4m3', 128)
    calls += [('channel', lambda: q.per_channel_cast(t, 'e4m3', 128, True)), ('transpose', lambda: q.per_channel_cast_and_transpose(t, 'e4m3', 32)),
              ('gather', lambda: q.per_channel_cast_fused(quantised, 'e4m3', 128, num_per_channels=128, pos_to_token=p2t)),
              ('swiglu channel', lambda: q.swiglu_forward_and_per_channel_cast_and_transpose(t, 'e4m3', 128, swiglu_clamp_value=1.5))]
    _compare(monkeypatch, calls)


@pytest.mark.gpu
def test_uninitialised_memory_is_filled_where_torch_is_told_to():
    """Three rows of column-major scales are stored in columns of four: the fourth is written by nobody but torch.empty."""
    import tilekernels_amd as tk
    x = _x(3, 512)
    torch.use_deterministic_algorithms(True)
    try:
        _, sf = tk.quant.per_token_cast(x, 'e4m3', 128, use_tma_aligned_col_major_sf=True)
    finally:
        torch.use_deterministic_algorithms(False)
    stored = torch.as_strided(sf, (4, 4), (4, 1))
    assert bool(stored[:, 3].isnan().all()) and torch.equal(stored[:, :3].T, sf)


@pytest.mark.gpu
def test_calls_the_python_code_takes(monkeypatch):
    """Empty inputs, modes, number types and options the native path leaves alone: the result is that of the Python code."""
    import tilekernels_amd as tk
    from torch.utils._python_dispatch import TorchDispatchMode
    q = tk.quant
    x = _x(8, 512)

    class Seen(TorchDispatchMode):
        calls = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Seen.calls += 1
            return func(*args, **(kwargs or {}))

    def in_mode():
        with Seen():
            return q.per_token_cast(x, 'e4m3', 128)

    _compare(monkeypatch, [('mode', in_mode), ('empty', lambda: q.per_token_cast(x[:0], 'e4m3', 128)),
                           ('options as numbers', lambda: q.per_token_cast(x, 'e4m3', 128, None, 1, 1, 1)),
                           ('integer clamp', lambda: q.swiglu_forward_and_per_token_cast(x, 'e4m3', 128, swiglu_clamp_value=2))], native=False)
    assert Seen.calls > 0
    for bad in (lambda: q.per_token_cast(x, 'e4m3', 48), lambda: q.per_token_cast(x, 'e3m4', 128), lambda: q.per_token_cast(x.half(), 'e4m3', 128),
                lambda: q.per_block_cast(x.T, 'e4m3', (128, 128)), lambda: q.per_token_cast(x, 'e4m3', 128, None, False, False, True),
                lambda: tk.moe.reduce_fused(x[:, :128], None, torch.zeros((1, 1), dtype=torch.int32, device='cuda'))):
        with pytest.raises(AssertionError):
            bad()
    from tilekernels_amd._ffi import TkError
    with pytest.raises(TkError):                     # misaligned rows
        q.per_token_cast(_x(8, 513)[:, 1:], 'e4m3', 128)


@pytest.mark.gpu
def test_watched_and_wrapped_calls_are_left_alone():
    """Tracing, function transforms, function modes and tensors that are more than their storage: the native functions return None."""
    from torch.overrides import TorchFunctionMode
    from tilekernels_amd import _ffi
    x = _x(8, 512, torch.float32)
    seen = []

    def native(v):
        seen.append(_ffi.host.per_token_cast(v, 'e4m3', 128, None, False, False, False))
        return v.sum()

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    def in_mode():
        with Mode():
            seen.append(_ffi.host.per_token_cast(x, 'e4m3', 128, None, False, False, False))

    def outer(v):       # a tensor from outside the transform
        seen.append(_ffi.host.per_token_cast(x, 'e4m3', 128, None, False, False, False))
        return v.sum()

    sub, negative = x.as_subclass(Sub), torch._neg_view(x)
    assert type(sub) is Sub and negative.is_neg()
    cases = {'trace': lambda: torch.jit.trace(native, x, check_trace=False), 'vmap': lambda: torch.func.vmap(native)(x[None]),
             'grad': lambda: torch.func.grad(native)(x), 'jvp': lambda: torch.func.jvp(native, (x,), (x,)),
             'functionalize': lambda: torch.func.functionalize(native)(x), 'inside vmap': lambda: torch.func.vmap(outer)(x),
             'inside grad': lambda: torch.func.grad(outer)(x), 'function mode': in_mode, 'subclass': lambda: native(sub),
             'negated view': lambda: native(negative), 'zero tensor': lambda: native(torch._efficientzerotensor((8, 512), device='cuda'))}
    for name, run in cases.items():
        seen.clear()
        native(x)
        run()
        native(x)
        assert len(seen) >= 3 and seen[0] is not None and seen[-1] is not None, name
        assert all(r is None for r in seen[1:-1]), name


@pytest.mark.gpu
def test_the_wait_for_segment_lengths_is_seen_by_sync_debug_mode():
    """A call that trims waits for the stream: torch refuses or reports that where it is told to, and has nothing to say to calls that do not wait."""
    import tilekernels_amd as tk
    from tilekernels_amd import _ffi
    idx = torch.randint(0, 8, (64, 4), generator=torch.Generator().manual_seed(3)).cuda()
    want = tk.moe.get_fused_mapping(idx, 8, 0, 16)
    assert _ffi.host.get_fused_mapping(idx, 8, 0, 16, False) is not None
    try:
        torch.cuda.set_sync_debug_mode('error')
        with pytest.raises(RuntimeError, match='synchroniz'):
            tk.moe.get_fused_mapping(idx, 8, 0, 16)
        for args in ((idx, 8, 512, 16, False), (idx, 8, 0, 16, True)):
            assert _ffi.host.get_fused_mapping(*args) is not None
        torch.cuda.set_sync_debug_mode('warn')
        with pytest.warns(UserWarning, match='synchroniz'):
            got = tk.moe.get_fused_mapping(idx, 8, 0, 16)
    finally:
        torch.cuda.set_sync_debug_mode('default')
    assert got[7] == want[7] and all(torch.equal(a, b) for a, b in zip(got[:7], want[:7]))


@pytest.mark.gpu
def test_threads_on_their_own_streams():
    """The lock is released around each launch: threads that call at the same time get the results each would get alone."""
    import threading
    import tilekernels_amd as tk
    g = torch.Generator().manual_seed(5)
    inputs, wants = [], []

    def calls(x, idx):
        m = tk.moe.get_fused_mapping(idx, 8, 1024, 16)
        e = tk.moe.expand_to_fused(x, m[3], m[0])
        c = tk.quant.per_token_cast(x, 'e4m3', 128, None, True, True, True)
        s = tk.quant.swiglu_forward_and_per_token_cast(e, 'e4m3', 128, pos_to_expert=m[0])
        r = tk.moe.reduce_fused(e, None, m[3])
        live = m[0] >= 0
        return [m[0], m[1], m[3], *c, s[0].view(torch.uint8)[live], s[1][live], e[live], r]

    for i in range(4):
        x = torch.randn((200 + i, 512), generator=g).to(torch.bfloat16).cuda()
        idx = torch.randint(-1, 8, (200 + i, 4), generator=g).cuda()
        inputs.append((x, idx))
        wants.append([_bytes(t) for t in calls(x, idx)])
    torch.cuda.synchronize()
    start, failed, finished = threading.Barrier(4), [], []

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            start.wait()
            for n in range(20):
                got = calls(*inputs[i])
                stream.synchronize()
                failed.extend((i, n, j) for j, (a, b) in enumerate(zip(got, wants[i])) if not torch.equal(_bytes(a), b))
        finished.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert sorted(finished) == [0, 1, 2, 3] and not failed, failed[:10]


@pytest.mark.parametrize('op', ['per_token_cast', 'per_block_cast', 'cast_back', 'swiglu_forward', 'reduce_fused', 'expand_to_fused', 'get_fused_mapping'])
def test_cpu_tensors_are_left_alone(op):
    from tilekernels_amd import _ffi
    x, sf = torch.zeros((4, 512), dtype=torch.bfloat16), torch.ones((4, 4))
    t2p, e = torch.zeros((4, 2), dtype=torch.int32), torch.zeros((8,), dtype=torch.int32)
    args = {'per_token_cast': (x, 'e4m3', 128, None, False, False, False), 'per_block_cast': (x, 'e4m3', (128, 128), False, False, False),
            'cast_back': ((x.to(torch.float8_e4m3fn), sf), 'bf16', 1, 128, None), 'reduce_fused': (x, None, t2p, '', None),
            'swiglu_forward': (x, 'e4m3', 128, None, None, None, False, False, False, None, None),
            'expand_to_fused': (x, None, None, t2p, e, False), 'get_fused_mapping': (t2p.long(), 8, 0, 16, False)}[op]
    fn = getattr(_ffi.host, op)
    assert fn(*args) is None
    assert fn(*[None] * len(args)) is None and fn(*[object()] * len(args)) is None
    with pytest.raises(TypeError):
        fn()


def test_native_path_is_named_for_what_it_was_built_against():
    import sysconfig
    from tilekernels_amd import _ffi
    name = os.path.basename(_ffi.HOST_PATH)
    assert torch.__version__ in name and sysconfig.get_config_var('SOABI') in name
    assert os.path.exists(_ffi.HOST_PATH)


@pytest.mark.parametrize('content', [None, b'not a library'], ids=['missing', 'unusable'])
def test_calls_without_a_native_path_are_left_to_python(monkeypatch, tmp_path, content):
    """A library built for another torch or Python is not loaded: one warning, then every call is that of the Python code."""
    import warnings
    import tilekernels_amd as tk
    from tilekernels_amd import _ffi
    path = tmp_path / '_host.so'
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(_ffi, 'HOST_PATH', str(path))
    monkeypatch.setattr(_ffi, 'host', _ffi._UnloadedHost())
    x = torch.zeros((4, 512), dtype=torch.bfloat16)
    with pytest.warns(RuntimeWarning, match='native call path'):
        with pytest.raises(_ffi.TkError, match='GPU only'):
            tk.quant.per_token_cast(x, 'e4m3', 128)
    with warnings.catch_warnings():
        warnings.simplefilter('error')
        with pytest.raises(_ffi.TkError, match='GPU only'):
            tk.quant.per_block_cast(x, 'e4m3', (128, 128))
        with pytest.raises(AssertionError):
            tk.quant.per_token_cast(x, 'e4m3', 48)


def test_native_path_is_loaded_once_by_threads(monkeypatch):
    import threading
    from tilekernels_amd import _ffi
    loads, load_host = [], _ffi._load_host
    monkeypatch.setattr(_ffi, '_load_host', lambda: loads.append(1) or load_host())
    monkeypatch.setattr(_ffi, 'host', _ffi._UnloadedHost())
    results = []
    threads = [threading.Thread(target=lambda: results.append(_ffi.host.cast_back(None, None, None, None, None))) for _ in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert results == [None] * 8 and len(loads) == 1
