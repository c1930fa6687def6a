"""The work a user of tilekernels_amd has it do, as cases that can be timed and compared.

A case is a dict of plain values; ``prepare`` builds on the GPU what a program holds before the call, ``run`` is one pass
through the public entry points, ``work`` the bytes and operations the pass cannot do without.  Eight kinds of pass:

* ``token_cast``      the per-token cast of activations or gradients (or of codes that are quantised already)
* ``round_trip``      a per-token cast and the dequantisation of what it gave: a cache or a message that is written and read
* ``block_cast``      the per-block cast of a weight matrix
* ``swiglu_cast``     the fused activation + cast of a dense feed-forward layer
* ``swiglu_backward`` the backward of that activation for the rows one expert-parallel rank holds
* ``wgrad_operands``  the two transposed operands of a feed-forward layer's weight gradient
* ``channel_requant`` the per-channel operand of an expert's weight gradient, gathered from the FP8 activations
* ``moe_layer``       what this package does around the two grouped products of a mixture-of-experts layer: quantise the tokens,
                      map and expand them, activation + cast between the products, weighted reduction back to tokens
"""
import math

import torch

import tilekernels_amd as tk

DEVICE = 'cuda'
LAYOUTS = ('row', 'col', 'packed')          # row-major fp32, column-major fp32, column-major packed UE8M0 scales


def listed():
    return [
        # one decoding step's activations for the next FP8 product: the launch and the host path count
        {'name': 'token_cast_decode', 'kind': 'token_cast', 'tokens': 64, 'hidden': 7168, 'source': 'bf16', 'fmt': 'e4m3',
         'group': 128, 'layout': 'row'},
        # a prefill batch of the same
        {'name': 'token_cast_prefill', 'kind': 'token_cast', 'tokens': 4096, 'hidden': 7168, 'source': 'bf16', 'fmt': 'e4m3',
         'group': 128, 'layout': 'row'},
        # a large batch to FP4 with packed power-of-two scales
        {'name': 'token_cast_fp4_large', 'kind': 'token_cast', 'tokens': 16384, 'hidden': 7168, 'source': 'bf16', 'fmt': 'e2m1',
         'group': 32, 'layout': 'packed'},
        # fp32 gradients, a token count that is no multiple of anything, column-major scales as a grouped product reads them
        {'name': 'token_cast_fp32_ragged', 'kind': 'token_cast', 'tokens': 4001, 'hidden': 2560, 'source': 'fp32', 'fmt': 'e4m3',
         'group': 128, 'layout': 'col'},
        # short rows (a compressed attention cache) written as FP8 with 1 x 64 scales and read back
        {'name': 'round_trip_short_rows', 'kind': 'round_trip', 'tokens': 8001, 'hidden': 576, 'source': 'bf16', 'fmt': 'e4m3',
         'group': 64, 'layout': 'row', 'back': 'bf16'},
        # a weight matrix, 128 x 128 blocks
        {'name': 'block_cast_weight', 'kind': 'block_cast', 'rows': 7168, 'cols': 2048, 'source': 'bf16', 'fmt': 'e4m3', 'block_m': 128,
         'block_k': 128, 'layout': 'row'},
        # the activation of a dense layer
        {'name': 'swiglu_cast_dense', 'kind': 'swiglu_cast', 'tokens': 8192, 'hidden': 2048, 'source': 'bf16', 'group': 128,
         'layout': 'row', 'clamp': False},
        # its backward on one of eight expert-parallel ranks
        {'name': 'swiglu_backward_rank', 'kind': 'swiglu_backward', 'sent': 4001, 'topk': 6, 'experts': 32, 'ranks': 8, 'hidden': 2048,
         'group': 128, 'align': 128, 'clamp': False},
        # weight gradient of the second product: activation recomputed and transposed, output gradient transposed
        {'name': 'wgrad_operands', 'kind': 'wgrad_operands', 'tokens': 8064, 'inner': 2048, 'hidden': 4096, 'group': 128, 'clamp': False},
        # weight gradient of the first product of the experts: FP8 tokens gathered into expert order, one scale per 128 rows
        {'name': 'channel_requant_gather', 'kind': 'channel_requant', 'sent': 1024, 'topk': 8, 'experts': 32, 'ranks': 8, 'hidden': 7168,
         'align': 128},
        # one decoding step of a layer on one of eight ranks, buffers of a fixed size (as a captured graph needs them)
        {'name': 'moe_layer_decode', 'kind': 'moe_layer', 'sent': 64, 'topk': 8, 'experts': 32, 'ranks': 8, 'hidden': 4096, 'inner': 2048,
         'align': 16, 'fixed': True, 'layout': 'row', 'weigh': 'reduce'},
        # a prefill or training batch of the same layer, buffers trimmed to what arrived
        {'name': 'moe_layer_prefill', 'kind': 'moe_layer', 'sent': 4096, 'topk': 8, 'experts': 32, 'ranks': 8, 'hidden': 7168, 'inner': 2048,
         'align': 128, 'fixed': False, 'layout': 'col', 'weigh': 'swiglu'},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _width(rng, step, low=512, high=11008):
    """A hidden size: one of the usual ones, or any multiple of `step`."""
    usual = [h for h in (576, 1024, 2048, 2560, 3072, 4096, 6144, 7168) if low <= h <= high and h % step == 0]
    return rng.choice(usual) if rng.random() < 0.6 else max(step, _log(rng, low, high) // step * step)


def _draw_kind(rng, kind):
    layout = rng.choice(LAYOUTS)
    ep = lambda: rng.choice([(32, 8), (9, 8), (4, 64), (256, 1), (72, 1)])        # experts of a rank, ranks
    if kind in ('token_cast', 'round_trip'):
        case = {'kind': kind, 'tokens': _log(rng, 1, 16384), 'hidden': _width(rng, 64), 'fmt': rng.choice(['e4m3', 'e4m3', 'e2m1']),
                'source': rng.choice(['bf16', 'bf16', 'bf16', 'fp32']), 'group': rng.choice([32, 64, 128, 128]), 'layout': layout}
        if kind == 'token_cast':
            if rng.random() < 0.15:
                case['source'] = 'e4m3'
        else:
            case['back'] = rng.choice(['bf16', 'bf16', 'fp32'])
            if rng.random() < 0.25:                                                # 12-bit codes, one scale per row
                case.update(fmt='e5m6', group=case['hidden'], layout='row')
        return case
    if kind == 'block_cast':
        return {'kind': kind, 'rows': _log(rng, 512, 16384), 'cols': _width(rng, 64), 'source': rng.choice(['bf16', 'bf16', 'fp32']),
                'fmt': rng.choice(['e4m3', 'e4m3', 'e2m1']), 'block_m': 128, 'block_k': rng.choice([128, 128, 32]), 'layout': layout}
    if kind == 'swiglu_cast':
        return {'kind': kind, 'tokens': _log(rng, 1, 32768), 'hidden': _width(rng, 128), 'source': rng.choice(['bf16', 'bf16', 'bf16', 'fp32']),
                'group': 128, 'layout': layout, 'clamp': rng.random() < 0.3}
    if kind == 'wgrad_operands':
        return {'kind': kind, 'tokens': 128 * _log(rng, 1, 128), 'inner': _width(rng, 128), 'hidden': _width(rng, 64),
                'group': rng.choice([32, 128, 128]), 'clamp': rng.random() < 0.3}
    experts, ranks = ep()
    case = {'kind': kind, 'sent': _log(rng, 16, 8192), 'topk': rng.choice([2, 6, 8, 9]), 'experts': experts, 'ranks': ranks}
    if experts * ranks < case['topk']:
        case['topk'] = 2
    if kind == 'swiglu_backward':
        case.update(hidden=_width(rng, 128), group=rng.choice([32, 128, 128]), align=rng.choice([64, 128]), clamp=rng.random() < 0.3)
    elif kind == 'channel_requant':
        case.update(hidden=_width(rng, 128), align=rng.choice([64, 128]))
    else:
        case.update(hidden=_width(rng, 256, 1024, 7168), inner=_width(rng, 128, 512, 4096), align=rng.choice([16, 64, 128]),
                    fixed=case['sent'] <= 512 and rng.random() < 0.5, layout=rng.choice(['row', 'col']),
                    weigh=rng.choice(['swiglu', 'reduce']))
    return case


def draw(rng):
    most = max(work(c)['bytes'] for c in listed())
    while True:
        case = _draw_kind(rng, rng.choice(['token_cast', 'round_trip', 'block_cast', 'swiglu_cast', 'swiglu_backward', 'wgrad_operands',
                                           'channel_requant', 'moe_layer']))
        if work(case)['bytes'] <= most and (case['kind'] not in ('swiglu_backward', 'channel_requant', 'moe_layer') or _pairs(case) >= 1):
            return case


# ---- routing -------------------------------------------------------------------------------------------------------------

def _pairs(case):
    """Expected (token, expert) pairs of one rank: every token of every rank chooses `topk` of all experts."""
    return case['sent'] * case['topk']


def _arrived(case):
    """Expected tokens of one rank: those with at least one of their experts here."""
    e, total, none = case['experts'], case['experts'] * case['ranks'], 1.0
    for i in range(case['topk']):
        none *= max(total - e - i, 0) / (total - i)
    return case['sent'] * case['ranks'] * (1 - none)


def _rows(case):
    """Expected expanded rows, the padding of every expert's segment among them: an expert's entries are close to Poisson
    distributed, and its segment has one block of `align` rows more for every multiple of `align` that they exceed."""
    mean, blocks = _pairs(case) / case['experts'], 0.0
    for j in range(int((mean + 8 * math.sqrt(mean)) / case['align']) + 1):
        blocks += 0.5 * math.erfc((j * case['align'] + 0.5 - mean) / math.sqrt(2 * mean)) if j else 1 - math.exp(-mean)
    return case['experts'] * case['align'] * blocks


def _route(case, g):
    """Expert ids (int64, -1 where the expert is on another rank) and weights of the tokens that reach this rank.

    How many tokens and rows arrive hangs on the case alone, so that every seed's outputs have the same shapes: one random
    routing is drawn for the case, and the seed decides the order of its tokens and of this rank's experts, and the weights."""
    n, e, k, ranks = case['sent'], case['experts'], case['topk'], case['ranks']
    base = torch.Generator(device=DEVICE).manual_seed(1)
    idx = torch.topk(torch.rand((n * ranks, e * ranks), generator=base, device=DEVICE), k=k, dim=-1, sorted=False).indices
    idx = idx.masked_fill(idx >= e, -1)
    idx = idx[(idx >= 0).any(dim=1)]
    if idx.shape[0] == 0:                          # a tiny batch that went elsewhere: one token stays
        idx = torch.full((1, k), -1, dtype=torch.int64, device=DEVICE)
        idx[0, 0] = 0
    experts = torch.cat([torch.randperm(e, generator=g, device=DEVICE), torch.full((1,), -1, dtype=torch.int64, device=DEVICE)])
    idx = experts[idx[torch.randperm(idx.shape[0], generator=g, device=DEVICE)]]      # index -1: the last entry, which is -1
    weights = torch.rand(idx.shape, generator=g, device=DEVICE) + 0.05
    return idx.contiguous(), (weights / weights.sum(-1, keepdim=True)).contiguous()


# ---- inputs --------------------------------------------------------------------------------------------------------------

def _normal(g, shape, dtype=torch.bfloat16, scale=1.0):
    return (torch.randn(shape, generator=g, device=DEVICE) * scale).to(dtype)


def _activations(g, shape, dtype=torch.bfloat16):
    """Normal values, one in a thousand a hundred times as large."""
    x = torch.randn(shape, generator=g, device=DEVICE)
    x.view(-1)[torch.randint(0, x.numel(), (max(1, x.numel() // 1000),), generator=g, device=DEVICE)] *= 100
    return x.to(dtype)


def _dtype(case):
    return torch.float32 if case['source'] == 'fp32' else torch.bfloat16


def _sf_options(layout):
    return {'row': {}, 'col': dict(use_tma_aligned_col_major_sf=True),
            'packed': dict(use_tma_aligned_col_major_sf=True, round_sf=True, use_packed_ue8m0=True)}[layout]


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    kind, state = case['kind'], {'case': case}
    if kind in ('token_cast', 'round_trip'):
        x = _activations(g, (case['tokens'], case['hidden']), _dtype(case))
        if case['source'] == 'e4m3':
            x = tk.quant.per_token_cast(x, 'e4m3', 128)
        state['x'] = x
    elif kind == 'block_cast':
        w = _normal(g, (case['rows'], case['cols']), torch.float32, 0.02)
        w[torch.randint(0, case['rows'], (16,), generator=g, device=DEVICE)] *= 50
        state['x'] = w.to(_dtype(case))
    elif kind == 'swiglu_cast':
        state['x'] = _normal(g, (case['tokens'], 2 * case['hidden']), _dtype(case), 2.0)
    elif kind == 'wgrad_operands':
        state['x'] = _normal(g, (case['tokens'], 2 * case['inner']), scale=2.0)
        state['grad'] = _normal(g, (case['tokens'], case['hidden']), scale=1e-3)
    else:
        idx, weights = _route(case, g)
        maps = tk.moe.get_fused_mapping(idx, case['experts'], 0, case['align'])
        rows, tokens = maps[0].shape[0], idx.shape[0]
        if kind == 'swiglu_backward':
            x = _normal(g, (rows, 2 * case['hidden']), scale=2.0)
            state.update(x=tk.quant.per_token_cast(x, 'e4m3', case['group']), grad=_normal(g, (rows, case['hidden']), scale=1e-2),
                         weights=weights, maps=maps)
        elif kind == 'channel_requant':
            x = _activations(g, (tokens, case['hidden']))
            state.update(x=tk.quant.per_token_cast(x, 'e4m3', 128), pos_to_token=maps[1])
        else:
            if case['fixed']:                      # the most rows that so many tokens can take
                rows = (idx.numel() + (case['align'] - 1) * case['experts']) // case['align'] * case['align']
            state.update(tokens=_activations(g, (tokens, case['hidden'])), idx=idx, weights=weights, rows=rows if case['fixed'] else 0,
                         first=_normal(g, (rows, 2 * case['inner']), scale=2.0),      # what the first grouped product gave
                         second=_normal(g, (rows, case['hidden'])))                    # what the second one gave
    return state


def run(state):
    case = state['case']
    kind = case['kind']
    if kind == 'token_cast':
        block = (1, 128) if case['source'] == 'e4m3' else None
        return tk.quant.per_token_cast(state['x'], case['fmt'], case['group'], block, **_sf_options(case['layout']))
    if kind == 'round_trip':
        codes = tk.quant.per_token_cast(state['x'], case['fmt'], case['group'], **_sf_options(case['layout']))
        special = 'e5m6' if case['fmt'] == 'e5m6' else None
        return codes, tk.quant.per_token_cast_back(codes, case['back'], case['group'], x_special_fmt=special)
    if kind == 'block_cast':
        return tk.quant.per_block_cast(state['x'], case['fmt'], (case['block_m'], case['block_k']), **_sf_options(case['layout']))
    if kind == 'swiglu_cast':
        return tk.quant.swiglu_forward_and_per_token_cast(state['x'], 'e4m3', case['group'], swiglu_clamp_value=7.0 if case['clamp'] else None,
                                                          **_sf_options(case['layout']))
    if kind == 'wgrad_operands':
        return (tk.quant.swiglu_forward_and_per_channel_cast_and_transpose(state['x'], 'e4m3', case['group'],
                                                                           swiglu_clamp_value=7.0 if case['clamp'] else None),
                tk.quant.per_channel_cast_and_transpose(state['grad'], 'e4m3', case['group']))
    if kind == 'swiglu_backward':
        _, _, pos_to_token_topk, token_topk_to_pos = state['maps'][:4]
        return tk.quant.swiglu_backward_and_per_token_cast(state['x'], state['grad'], state['weights'], pos_to_token_topk, token_topk_to_pos,
                                                           case['group'], swiglu_clamp_value=7.0 if case['clamp'] else None)
    if kind == 'channel_requant':
        return tk.quant.per_channel_cast_fused(state['x'], 'e4m3', 128, num_per_channels=128, pos_to_token=state['pos_to_token'])
    sf = _sf_options(case['layout'])
    weights = state['weights']
    maps = tk.moe.get_fused_mapping(state['idx'], case['experts'], state['rows'], case['align'])
    pos_to_expert, pos_to_token, pos_to_token_topk, token_topk_to_pos = maps[:4]
    tokens = tk.quant.per_token_cast(state['tokens'], 'e4m3', 128)
    expanded = tk.moe.expand_to_fused_with_sf(tokens, 128, token_topk_to_pos, pos_to_expert, **sf)
    if case['weigh'] == 'swiglu':
        act = tk.quant.swiglu_forward_and_per_token_cast(state['first'], 'e4m3', 128, pos_to_token_topk, weights, pos_to_expert, **sf)
        out = tk.moe.reduce_fused(state['second'], None, token_topk_to_pos)
    else:
        act = tk.quant.swiglu_forward_and_per_token_cast(state['first'], 'e4m3', 128, pos_to_expert=pos_to_expert, **sf)
        out = tk.moe.reduce_fused(state['second'], weights, token_topk_to_pos)
    return maps[:7], tokens, expanded, act, out


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------

_BITS = {'bf16': 16, 'fp32': 32, 'e4m3': 8, 'e2m1': 4, 'e5m6': 12}


def _sf_bytes(rows, cols, group, layout='row'):
    return rows * math.ceil(cols / group) * (1 if layout == 'packed' else 4)


def work(case):
    kind = case['kind']
    if kind in ('token_cast', 'round_trip'):
        n = case['tokens'] * case['hidden']
        sf = _sf_bytes(case['tokens'], case['hidden'], case['group'], case['layout'])
        b = n * (_BITS[case['source']] + _BITS[case['fmt']]) / 8 + sf
        f = 3.0 * n                                                      # maximum, product, rounding
        if case['source'] == 'e4m3':
            b, f = b + _sf_bytes(case['tokens'], case['hidden'], 128), f + n
        if kind == 'round_trip':
            b, f = b + n * (_BITS[case['fmt']] + _BITS[case['back']]) / 8 + sf, f + n
    elif kind == 'block_cast':
        n = case['rows'] * case['cols']
        b = n * (_BITS[case['source']] + _BITS[case['fmt']]) / 8 + _sf_bytes(math.ceil(case['rows'] / case['block_m']), case['cols'], case['block_k'],
                                                                              case['layout'])
        f = 3.0 * n
    elif kind == 'swiglu_cast':
        n = case['tokens'] * case['hidden']
        b = n * (2 * _BITS[case['source']] / 8 + 1) + _sf_bytes(case['tokens'], case['hidden'], case['group'], case['layout'])
        f = 8.0 * n
    elif kind == 'wgrad_operands':
        a, d = case['tokens'] * case['inner'], case['tokens'] * case['hidden']
        b = a * 5 + d * 3 + _sf_bytes(case['tokens'] // case['group'], case['inner'] + case['hidden'], 1)
        f = 8.0 * a + 3.0 * d
    elif kind == 'swiglu_backward':
        r, p, h = _rows(case), _pairs(case), case['hidden']             # rows of padding are written, not read
        b = p * h * (2 + 2) + r * h * (2 + 2 + 4) + _sf_bytes(p + r, 2 * h, case['group']) + 4 * r + 12 * _arrived(case) * case['topk']
        f = 24.0 * _pairs(case) * h
    elif kind == 'channel_requant':
        r, t, h = _rows(case), _arrived(case), case['hidden']
        b = t * h + r * h + _sf_bytes(t, h, 128) + _sf_bytes(r / 128, h, 1) + 4 * r
        f = 4.0 * r * h
    else:
        r, t, p, h, i = _rows(case), _arrived(case), _pairs(case), case['hidden'], case['inner']
        b = t * case['topk'] * (8 + 4) + 12 * r                          # the mapping
        b += t * h * 3 + _sf_bytes(t, h, 128)                            # the tokens' cast
        b += t * h + r * h + _sf_bytes(t + r, h, 128)                    # the expansion
        b += p * 4 * i + r * i + _sf_bytes(r, i, 128)                    # activation + cast
        b += p * 2 * h + t * 2 * h + 8 * t * case['topk']                # the reduction
        f = 3.0 * t * h + 8.0 * p * i + 2.0 * p * h
    return {'bytes': float(b), 'flops': float(f)}


def tolerance(case):
    """Casts, dequantisation and index lists are whole-number results: bit for bit.  Where an exponential precedes the
    rounding, a value on a rounding boundary may take the neighbouring code, an eighth of it away.  Against float64
    evaluations 4e-7 to 2.5e-6 of the codes do in the forward (2-norm of the difference up to 2.5e-4) and 1.4e-5 in the backward
    (6.5e-4); scales and fp32 gradients are within 8e-8 and 1.1e-7, bf16 results within 2.2e-5."""
    if case['kind'] in ('token_cast', 'round_trip', 'block_cast', 'channel_requant'):
        return 'exact'
    return {'rel': 2.6e-3 if case['kind'] == 'swiglu_backward' else 1e-3, 'max': 0.13}
