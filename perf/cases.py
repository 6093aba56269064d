"""The calls whose speed this package is judged by, as a program that serves
the model makes them.

Each case is one pass through the public entry points: a model session's step
(`AttentionKV`), the fused attention layer (`attention_fused`), the raw GQA
core (`attention`) and the paged cache's import and export (`PagedKV.pack` and
`unpack`).  `listed()` names the typical calls, `draw()` gives further ones of
the same ranges, `prepare()` makes what the program holds before the call,
`run()` is the call, `work()` what it cannot do without, `exact()` the same
results from plain torch in float64, and `tolerance()` how far another correct
implementation at the same precision may be from them.
"""
import math

import torch

from redshift_amd import attention as A
from redshift_amd.kvcache import AttentionKV

# The model's full-attention geometry (query heads, KV heads, head dim), and
# the smaller and the common 128-dim GQA geometries that the raw core takes.
MODEL = (24, 4, 256)
GEOMETRIES = (MODEL, (8, 2, 128), (32, 8, 128))
CONTEXT = 139264
EPSILON = 1e-6
MOST_FLOPS = 4 * 256 * 24 * (2048 * 6144 + 2048 * 2049 // 2)


def _case(name, kind, tokens, position, geometry=MODEL, dtype='f16', layers=1, outliers=0):
    c = {'kind': kind, 'tokens': tokens, 'position': position, 'q_heads': geometry[0], 'kv_heads': geometry[1],
         'head_dim': geometry[2], 'dtype': dtype, 'layers': layers, 'outliers': outliers}
    if name:
        c['name'] = name
    return c


def listed():
    return [
        # A chat's first verification steps: the prompt is a few words long,
        # so launches and latency are all there is.  Four layers of a session.
        _case('session_verify8_100', 'session', 8, 100, layers=4),
        # Token by token after a prompt of a few pages (ragged length).
        _case('session_decode_5k', 'session', 1, 5003, layers=4),
        # Speculative verification in a long conversation: the common step of
        # a server with draft tokens.
        _case('session_verify8_16k', 'session', 8, 16384, layers=4),
        # A short follow-up message (64 tokens) appended to a long context.
        _case('fused_chunk64_16k', 'fused', 64, 16384),
        # One chunk of a long prompt's prefill, in the model's fused layer.
        _case('fused_chunk2048_6k', 'fused', 2048, 6144),
        # One token at the full context: a few keys dominate.
        _case('fused_decode_139k', 'fused', 1, 139263, outliers=64),
        # The raw core as a caller with its own preparation uses it: decode,
        # verification and a prompt chunk of a bf16 model.
        _case('raw_decode_4k', 'raw', 1, 4095),
        _case('raw_verify8_16k', 'raw', 8, 16384),
        _case('raw_chunk2048_6k_bf16', 'raw', 2048, 6144, dtype='bf16'),
        # The common 128-dim GQA model: decode, and a whole ragged prompt.
        _case('gqa128_decode_9k_bf16', 'raw', 1, 9001, (32, 8, 128), 'bf16'),
        _case('gqa128_prompt_3000', 'raw', 3000, 0, (32, 8, 128)),
        # A prompt's token-major cache taken into pages and given back (a
        # prefix store, or another program's cache).
        _case('kv_import_export_20k', 'kv', 20001, 0),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _chunk(rng, geometry, most_tokens):
    """A prompt chunk: 9 tokens up, on a prefix of any length that keeps the
    call within the largest listed one."""
    tokens = _log(rng, 9, most_tokens)
    position = _log(rng, 1, 20000) - 1
    most = MOST_FLOPS // (4 * geometry[2] * geometry[0])
    return tokens, max(0, min(position, (most - tokens * (tokens + 1) // 2) // tokens))


def draw(rng):
    kind = rng.choice(('session', 'fused', 'fused_chunk', 'raw', 'raw_chunk', 'kv'))
    dtype = rng.choice(('f16', 'bf16'))
    geometry = rng.choice(GEOMETRIES)
    if kind == 'session':
        return _case(None, kind, rng.randint(1, 8), _log(rng, 16, 30000), layers=rng.randint(1, 4))
    if kind == 'fused':
        return _case(None, kind, rng.randint(1, 8), _log(rng, 16, CONTEXT - 8), outliers=rng.choice((0, 16)))
    if kind == 'fused_chunk':
        return _case(None, 'fused', *_chunk(rng, MODEL, 2048))
    if kind == 'raw':
        return _case(None, kind, rng.randint(1, 8), _log(rng, 16, CONTEXT - 8), geometry, dtype,
                     outliers=rng.choice((0, 16)))
    if kind == 'raw_chunk':
        return _case(None, 'raw', *_chunk(rng, geometry, 4096), geometry, dtype)
    return _case(None, kind, _log(rng, 30, 60000), 0, geometry, dtype)


# ---- what a program holds before the call ----------------------------------
def _generator(seed):
    return torch.Generator('cuda').manual_seed(seed)


def _normal(gen, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=gen, device='cuda', dtype=torch.float32) * std).to(dtype)


def _dtype(case):
    return torch.bfloat16 if case['dtype'] == 'bf16' else torch.float16


def _inputs(case, seed):
    """Per layer: the cached rows and the call's own tensors, from the seed."""
    gen = _generator(seed)
    hq, hkv, d = case['q_heads'], case['kv_heads'], case['head_dim']
    tokens, position, dtype = case['tokens'], case['position'], _dtype(case)
    layers = []
    for _ in range(case['layers']):
        raw = case['kind'] in ('raw', 'kv')
        keys = position + tokens if raw else position
        x = {'k_rows': _normal(gen, keys, hkv, d, std=.5, dtype=dtype),
             'v_rows': _normal(gen, keys, hkv, d, std=.5, dtype=dtype)}
        if case['outliers']:
            at = torch.randperm(keys, generator=gen, device='cuda')[:case['outliers']]
            x['k_rows'][at] *= 8
        if case['kind'] == 'raw':
            x['q'] = _normal(gen, tokens, hq, d, dtype=dtype)
        elif not raw:
            x['q_gate'] = _normal(gen, tokens, hq, 2 * d)
            x['key'] = _normal(gen, tokens, hkv, d)
            x['value'] = _normal(gen, tokens, hkv, d, std=.5)
            x['q_norm'] = 1 + .25 * _normal(gen, d)
            x['k_norm'] = 1 + .25 * _normal(gen, d)
        layers.append(x)
    return layers


def _fill(cache, x):
    """The cached rows in their pages; slots behind them hold zeros."""
    cache.k.zero_()
    cache.v.zero_()
    if x['k_rows'].shape[0]:
        cache.pack(x['k_rows'], x['v_rows'])


LAYER_INPUTS = ('q_gate', 'key', 'value', 'q_norm', 'k_norm')


def prepare(case, seed):
    layers = _inputs(case, seed)
    end = case['position'] + case['tokens']
    if case['kind'] == 'session':
        session = AttentionKV(case['layers'], context=end, epsilon=EPSILON)
        for cache, x in zip(session.caches, layers):
            _fill(cache, x)
        session.position = case['position']
        return {'case': case, 'session': session, 'inputs': [[x[n] for n in LAYER_INPUTS] for x in layers]}
    x = layers[0]
    cache = A.PagedKV(case['kv_heads'], case['head_dim'], A.round_capacity(end), _dtype(case))
    if case['kind'] == 'kv':
        cache.k.zero_()
        cache.v.zero_()
        return {'case': case, 'cache': cache, 'k_rows': x['k_rows'], 'v_rows': x['v_rows']}
    _fill(cache, x)
    if case['kind'] == 'fused':
        ws = A.workspace(A.fused_workspace_bytes(case['tokens'], case['position']))
        return {'case': case, 'cache': cache, 'inputs': [x[n] for n in LAYER_INPUTS], 'ws': ws}
    ws = A.workspace(A.attention_workspace_bytes(case['q_heads'], case['kv_heads'], case['head_dim'], case['tokens'],
                                                 case['position']))
    return {'case': case, 'cache': cache, 'q': x['q'], 'ws': ws}


# ---- the call ---------------------------------------------------------------
def run(state):
    case = state['case']
    if case['kind'] == 'session':
        # A verification whose tokens are all rejected: the session is where
        # it was, so the step can be repeated.
        session = state['session']
        session.begin(case['tokens'], recording=True)
        outs = [session.attend(i, *inputs) for i, inputs in enumerate(state['inputs'])]
        session.end()
        session.commit(0)
        return {'out': outs, 'k': [c.k for c in session.caches], 'v': [c.v for c in session.caches]}
    cache = state['cache']
    if case['kind'] == 'fused':
        out = A.attention_fused(*state['inputs'], cache, case['position'], EPSILON, ws=state['ws'])
        return {'out': out, 'k': cache.k, 'v': cache.v}
    if case['kind'] == 'raw':
        return {'out': A.attention(state['q'], cache, case['position'], 1 / math.sqrt(case['head_dim']),
                                   ws=state['ws'])}
    cache.pack(state['k_rows'], state['v_rows'])
    k_rows, v_rows = cache.unpack(0, case['tokens'])
    return {'k': cache.k, 'v': cache.v, 'k_rows': k_rows, 'v_rows': v_rows}


def work(case):
    hq, hkv, d = case['q_heads'], case['kv_heads'], case['head_dim']
    tokens, position = case['tokens'], case['position']
    row = 2 * hkv * d * 2          # K and V of one token
    if case['kind'] == 'kv':
        return {'bytes': 4 * tokens * row, 'flops': 0}     # rows to pages and back, read and written
    pairs = tokens * position + tokens * (tokens + 1) // 2
    flops = 4 * d * hq * pairs
    if case['kind'] == 'raw':
        moved = (position + tokens) * row + 2 * tokens * hq * d * 2
    else:
        # q, gate and output, key and value in fp32; the appended rows written.
        moved = position * row + tokens * (3 * hq * d * 4 + 2 * hkv * d * 4 + row)
    return {'bytes': case['layers'] * moved, 'flops': case['layers'] * flops}


def tolerance(case):
    if case['kind'] == 'kv':
        return 'exact'
    if case['kind'] == 'raw':
        # The output's own 16-bit rounding and that of the 16-bit weights:
        # 1.7e-3 (bf16) and 2.6e-4 .. 3.7e-4 (fp16) from float64.
        return {'rel': 7e-3 if case['dtype'] == 'bf16' else 1.5e-3}
    # fp32 queries and weights on an fp16 cache, fp32 output: 2e-7, and up to
    # 7.7e-6 where a new key rounds to the other fp16 neighbour.
    return {'rel': 3e-5}


# ---- the same in float64, from plain torch ---------------------------------
def _k_pages(rows, capacity):
    """Token-major [n, heads, d] as K pages: per head and 16 tokens, [d/8][16][8]."""
    n, heads, d = rows.shape
    full = torch.zeros(capacity, heads, d, dtype=rows.dtype, device=rows.device)
    full[:n] = rows
    return full.view(capacity // 16, 16, heads, d // 8, 8).permute(2, 0, 3, 1, 4).reshape(-1)


def _v_pages(rows, capacity):
    """Token-major [n, heads, d] as V pages: per head and 32 tokens (a, g, i),
    [d/16][g][16 dims][a][i]."""
    n, heads, d = rows.shape
    full = torch.zeros(capacity, heads, d, dtype=rows.dtype, device=rows.device)
    full[:n] = rows
    return full.view(capacity // 32, 2, 4, 4, heads, d // 16, 16).permute(4, 0, 5, 2, 6, 1, 3).reshape(-1)


def _attend(q, k, v, position, scale):
    """Causal GQA in float64: q [t, hq, d], k and v [n, hkv, d]; row t sees
    keys 0..position+t."""
    tokens, hq, d = q.shape
    hkv = k.shape[1]
    group = hq // hkv
    out = torch.empty(tokens, hq, d, dtype=torch.float64, device=q.device)
    at = torch.arange(k.shape[0], device=q.device)
    block = max(1, (1 << 26) // (group * k.shape[0]))
    for h in range(hkv):
        kt, vh = k[:, h].double().t().contiguous(), v[:, h].double().contiguous()
        for t0 in range(0, tokens, block):
            rows = q[t0:t0 + block, h * group:(h + 1) * group].double()
            b = rows.shape[0]
            s = (rows.reshape(b * group, d) @ kt).mul_(scale).view(b, group, -1)
            last = position + t0 + torch.arange(b, device=q.device)
            s.masked_fill_(at[None, None, :] > last[:, None, None], -math.inf)
            p = torch.softmax(s, -1)
            out[t0:t0 + b, h * group:(h + 1) * group] = (p.view(b * group, -1) @ vh).view(b, group, d)
    return out


def _norm_rope(x, weight, position):
    """RMSNorm times weight, then rotary position on the first 64 dims (pairs
    i, i + 32, base 1e7), in float64."""
    x, weight = x.double(), weight.double()
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPSILON) * weight
    t = torch.arange(x.shape[0], device=x.device, dtype=torch.float64) + position
    angle = t[:, None] * 1e7 ** (-torch.arange(32, device=x.device, dtype=torch.float64) / 32)
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., :32].clone(), x[..., 32:64].clone()
    x[..., :32], x[..., 32:64] = a * c - b * s, a * s + b * c
    return x


def _layer(case, x):
    d, position = case['head_dim'], case['position']
    q = _norm_rope(x['q_gate'][..., :d], x['q_norm'], position)
    new_k, new_v = _norm_rope(x['key'], x['k_norm'], position), x['value'].double()
    # The cache holds fp16: later rows attend to the rounded values.
    k = torch.cat([x['k_rows'], new_k.half()])
    v = torch.cat([x['v_rows'], new_v.half()])
    out = _attend(q, k, v, position, 1 / math.sqrt(d)) * torch.sigmoid(x['q_gate'][..., d:].double())
    capacity = A.PAGE_TOKENS * -(-k.shape[0] // A.PAGE_TOKENS)
    return (out, _k_pages(torch.cat([x['k_rows'].double(), new_k]), capacity),
            _v_pages(torch.cat([x['v_rows'].double(), new_v]), capacity))


def exact(case, seed):
    layers = _inputs(case, seed)
    x = layers[0]
    if case['kind'] == 'kv':
        return None
    if case['kind'] == 'raw':
        return {'out': _attend(x['q'], x['k_rows'], x['v_rows'], case['position'], 1 / math.sqrt(case['head_dim']))}
    done = [_layer(case, x) for x in layers]
    if case['kind'] == 'fused':
        return dict(zip(('out', 'k', 'v'), done[0]))
    return {n: [r[i] for r in done] for i, n in enumerate(('out', 'k', 'v'))}
