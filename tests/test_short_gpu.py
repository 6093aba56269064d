"""The one-launch fused kernel (up to 8 tokens on at most 256 keys) against the
oracle where its page and slot counts change: no cached page, one (from one
key to all 32), seven and eight (the new keys' page on a wave of its own, then
on wave 0 after its cached page), the last position; NaN past the prefix.
Tolerances of the reference's own test: output 3e-4, K 2e-3, V exact."""
import numpy as np
import pytest

from oracle import attention_ref as ref
from redshift_amd import attention as A
from tests.test_attention_gpu import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('batch,position', [(1, 0), (8, 0), (8, 1), (5, 31), (8, 32), (3, 33), (8, 224), (8, 225),
                                            (8, 248), (1, 255), (2, 193)])
def test_short_context_against_oracle(gpu, batch, position):
    torch = gpu
    rng = np.random.default_rng(100 * batch + position)
    kc, vc = ((rng.standard_normal((position, 4, 256)) * .5).astype(np.float16) for _ in 'kv')
    host = [rng.standard_normal(s).astype(np.float32) for s in ((batch, 24, 512), (batch, 4, 256), (batch, 4, 256))]
    host += [(1 + .25 * rng.uniform(-1, 1, 256)).astype(np.float32) for _ in 'qk']
    expected = ref.fused_attention(kc, vc, *host, batch, position, 1e-6)
    cache = A.PagedKV(4, 256, 256, torch.float16)
    cache.k.fill_(float('nan'))
    cache.v.fill_(float('nan'))
    if position:
        cache.pack(torch.from_numpy(kc).cuda(), torch.from_numpy(vc).cuda())
    out = A.attention_fused(*[torch.from_numpy(x).cuda() for x in host], cache, position, 1e-6)
    got = [out, *cache.unpack(0, position + batch)]
    torch.cuda.synchronize()
    for g, e, tolerance in zip(got, expected, (3e-4, 2e-3, 0)):
        assert_close(g.float().cpu().numpy(), e, tolerance)
