"""The front end's native calls against its Python route (which a tensor
subclass takes, and what else needs Python): the same bits for every option, the
caller's own output tensor back, the current stream, and the same errors.  Every
comparison first shows that its Python leg is one."""
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
    """t as a tensor subclass (nn.Parameter is none to the native calls)."""
    import torch

    class Subclass(torch.Tensor):
        pass
    return t.as_subclass(Subclass)


def native(name, *args):
    """The native call; None for what it does not take."""
    front = A._FRONT or A._load_front()
    assert front is not A._PythonRoute
    return getattr(front, name)(*args)


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

    def options():
        fresh = dict(kw)
        if 'out' in kw:
            fresh['out'] = torch.full_like(kw['out'], float('nan'))
        return fresh, (fresh.get('out'), fresh.get('ws'), fresh.get('out_dtype'))

    fresh, rest = options()
    want = native('attention', q, cache, 700, 1 / 16, *rest)
    assert want is not None and (want is fresh['out'] if 'out' in kw else True)
    assert native('attention', torch.nn.Parameter(q, requires_grad=False), cache, 700, 1 / 16, *rest) is not None
    wide = torch.zeros(5, 24, 512, dtype=q.dtype, device='cuda')
    wide[..., ::2] = q
    for query in (python_route(q), wide[..., ::2]):
        fresh, rest = options()
        assert native('attention', query, cache, 700, 1 / 16, *rest) is None
        got = A.attention(query, cache, 700, 1 / 16, **fresh)
        assert got is fresh['out'] if 'out' in kw else type(got) is torch.Tensor
        assert got.dtype == want.dtype and got.shape == want.shape and torch.equal(got, want)


def test_what_only_python_takes(gpu):
    """An integer scale, a subclass as output, workspace or cache tensor."""
    torch = gpu
    cache, q = make(torch, torch.float16)
    ws = A.workspace(A.attention_workspace_bytes(24, 4, 256, 5, 700))
    want = native('attention', q, cache, 700, 1.0, None, None, None)
    out = python_route(torch.zeros_like(q))
    for scale, o, w in ((1, None, None), (1.0, out, None), (1.0, None, python_route(ws))):
        assert native('attention', q, cache, 700, scale, o, w, None) is None
        assert torch.equal(A.attention(q, cache, 700, scale, out=o, ws=w).as_subclass(torch.Tensor), want)
    cache.k = python_route(cache.k)
    assert native('attention', q, cache, 700, 1.0, None, None, None) is None
    assert torch.equal(A.attention(q, cache, 700, 1.0), want)


@pytest.mark.parametrize('tokens,position', [(1, 0), (3, 40), (2, 700), (8, 700), (40, 700)])
def test_fused_routes_agree(gpu, tokens, position):
    torch = gpu
    g = torch.Generator('cuda').manual_seed(tokens)
    inputs = [torch.randn(s, generator=g, device='cuda') for s in ((tokens, 24, 512), (tokens, 4, 256),
                                                                    (tokens, 4, 256), (256,), (256,))]
    side = torch.cuda.Stream()
    outs = []
    for route in ('native', 'stream', 'python', 'subclass key', 'unaligned'):
        cache, _ = make(torch, torch.float16, tokens, position)
        x = list(inputs)
        if route == 'python':
            x[0] = python_route(x[0])
        if route == 'subclass key':
            x[1] = python_route(x[1])
        if route == 'unaligned':   # 4 bytes off a 16-byte boundary: copied in Python
            buf = torch.zeros(x[1].numel() + 1, device='cuda')
            buf[1:] = x[1].reshape(-1)
            x[1] = buf[1:].view(x[1].shape)
        assert (native('attention_fused', *x, cache, position, 1e-6, None, None) is None) == (
            route in ('python', 'subclass key', 'unaligned'))
        cache, _ = make(torch, torch.float16, tokens, position)   # as it was before that call
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
        rest = [args.get(n) for n in ('out', 'ws', 'out_dtype')]
        assert native('attention', python_route(q), cache, args['position'], args['scale'], *rest) is None
        if kind is RuntimeError:   # an error of the library: from either route
            with pytest.raises(kind, match=match):
                native('attention', q, cache, args['position'], args['scale'], *rest)
        else:
            assert native('attention', q, cache, args['position'], args['scale'], *rest) is None
    with pytest.raises(ValueError, match='q is torch.bfloat16'):
        A.attention(q.bfloat16(), cache, 700, 1 / 16)
    x = [torch.zeros(s, device='cuda') for s in ((2, 24, 512), (2, 4, 256), (2, 4, 256), (256,), (256,))]
    with pytest.raises(RuntimeError, match='epsilon must be finite and positive'):
        A.attention_fused(*x, cache, 3, -1.0)
    with pytest.raises(RuntimeError, match='attention context exceeds 139264'):
        A.attention_fused(*x, cache, 139263, 1e-6)
    with pytest.raises(ValueError, match='key must hold'):
        A.attention_fused(x[0], x[1][:1], *x[2:], cache, 3, 1e-6)
