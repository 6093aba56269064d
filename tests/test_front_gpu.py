"""The front end's native calls against its Python route (which a tensor
subclass takes): the same bits for every option, the caller's own output
tensor back, the current stream, and the same errors."""
import pytest

from redshift_amd import attention as A

pytestmark = pytest.mark.gpu


def make(torch, dtype, tokens=5, position=700, seed=0):
    g = torch.Generator('cuda').manual_seed(seed)
    cache = A.PagedKV(4, 256, A.round_capacity(position + tokens), dtype)
    cache.k.zero_()
    cache.v.zero_()
    rows = [torch.randn(position + tokens, 4, 256, generator=g, device='cuda').to(dtype) for _ in 'kv']
    cache.pack(*rows)
    return cache, torch.randn(tokens, 24, 256, generator=g, device='cuda').to(dtype)


def python_route(t):
    import torch
    return torch.nn.Parameter(t, requires_grad=False)


@pytest.mark.parametrize('dtype', ['float16', 'bfloat16'])
@pytest.mark.parametrize('out', ['none', 'given', 'float32', 'given float32'])
@pytest.mark.parametrize('ws', [False, True])
def test_attention_routes_agree(gpu, dtype, out, ws):
    torch = gpu
    cache, q = make(torch, getattr(torch, dtype))
    kw = {}
    if ws:
        kw['ws'] = A.workspace(A.attention_workspace_bytes(24, 4, 256, 5, 700))
    if out.startswith('given'):
        kw['out'] = torch.zeros(q.shape, dtype=torch.float32 if 'float32' in out else q.dtype, device='cuda')
    elif out == 'float32':
        kw['out_dtype'] = torch.float32
    native = A._load_front().attention(q, cache, 700, 1 / 16, kw.get('out'), kw.get('ws'), kw.get('out_dtype'))
    assert native is not None and (native is kw['out'] if 'out' in kw else True)
    native = native.clone()
    other = A.attention(python_route(q), cache, 700, 1 / 16, **kw)
    assert native.dtype == other.dtype and native.shape == other.shape and torch.equal(native, other)
    # A strided query takes the Python route (a copy); so does an int scale.
    wide = torch.zeros(5, 24, 512, dtype=q.dtype, device='cuda')
    wide[..., ::2] = q
    assert A._load_front().attention(wide[..., ::2], cache, 700, 1 / 16, None, None, None) is None
    assert torch.equal(A.attention(wide[..., ::2], cache, 700, 1 / 16, **kw), native)


@pytest.mark.parametrize('tokens,position', [(1, 0), (3, 40), (2, 700), (8, 700), (40, 700)])
def test_fused_routes_agree(gpu, tokens, position):
    torch = gpu
    g = torch.Generator('cuda').manual_seed(tokens)
    inputs = [torch.randn(s, generator=g, device='cuda') for s in ((tokens, 24, 512), (tokens, 4, 256),
                                                                    (tokens, 4, 256), (256,), (256,))]
    side = torch.cuda.Stream()
    outs = []
    for route in ('native', 'stream', 'python', 'unaligned'):
        cache, _ = make(torch, torch.float16, tokens, position)
        x = list(inputs)
        if route == 'python':
            x[0] = python_route(x[0])
        if route == 'unaligned':   # 4 bytes off a 16-byte boundary: copied in Python
            buf = torch.zeros(x[1].numel() + 1, device='cuda')
            buf[1:] = x[1].reshape(-1)
            x[1] = buf[1:].view(x[1].shape)
        torch.cuda.synchronize()
        with torch.cuda.stream(side if route == 'stream' else torch.cuda.current_stream()):
            outs.append(A.attention_fused(*x, cache, position, 1e-6))
        torch.cuda.synchronize()
        outs[-1] = (outs[-1], cache.k, cache.v)
    for o in outs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(o, outs[0]))


def test_errors_are_the_python_ones(gpu):
    torch = gpu
    cache, q = make(torch, torch.float16)
    for kw, kind, match in (({'position': -1}, RuntimeError, 'position must be non-negative'),
                            ({'position': 10 ** 6}, RuntimeError, 'exceeds the cache capacity'),
                            ({'scale': float('inf')}, RuntimeError, 'scale must be finite'),
                            ({'ws': torch.empty(16, dtype=torch.uint8, device='cuda')}, RuntimeError, 'workspace too small'),
                            ({'ws': torch.empty(1 << 26, dtype=torch.uint8)}, ValueError, 'workspace is on cpu'),
                            ({'out': torch.empty(5, 24, 256, device='cuda').bfloat16()}, ValueError, 'out must be'),
                            ({'out_dtype': torch.float64}, ValueError, 'out must be')):
        args = {'position': 700, 'scale': 1 / 16, **kw}
        for query in (q, python_route(q)):
            with pytest.raises(kind, match=match):
                A.attention(query, cache, **args)
    with pytest.raises(ValueError, match='q is torch.bfloat16'):
        A.attention(q.bfloat16(), cache, 700, 1 / 16)
    x = [torch.zeros(s, device='cuda') for s in ((2, 24, 512), (2, 4, 256), (2, 4, 256), (256,), (256,))]
    with pytest.raises(RuntimeError, match='epsilon must be finite and positive'):
        A.attention_fused(*x, cache, 3, -1.0)
    with pytest.raises(RuntimeError, match='attention context exceeds 139264'):
        A.attention_fused(*x, cache, 139263, 1e-6)
    with pytest.raises(ValueError, match='key must hold'):
        A.attention_fused(x[0], x[1][:1], *x[2:], cache, 3, 1e-6)
