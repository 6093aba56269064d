"""qv_kv_pack / qv_kv_unpack against the host page layout, bit for bit: ranges
that start and end inside a page (the page's other slots keep their values),
whole pages, one side alone, several KV heads, and buffers that are not
16-byte aligned (the value-by-value route)."""
import ctypes as ct

import numpy as np
import pytest

from redshift_amd import layout
from redshift_amd.runtime import check, library

pytestmark = pytest.mark.gpu


def _offset(torch, host, shift):
    """host as device memory that starts `shift` values past an aligned address."""
    buf = torch.zeros(host.size + 8, dtype=torch.int16, device='cuda')
    assert buf.data_ptr() % 16 == 0
    view = buf[shift:shift + host.size]
    view.copy_(torch.from_numpy(host.reshape(-1).view(np.int16)))
    return view


@pytest.mark.parametrize('sides', ['kv', 'k', 'v'])
@pytest.mark.parametrize('shift', [0, 1])
@pytest.mark.parametrize('kv_heads,head_dim,capacity,first,count', [
    (4, 256, 32, 0, 32), (1, 128, 32, 31, 1), (4, 256, 96, 5, 70), (3, 128, 160, 32, 96),
    (8, 128, 128, 17, 16), (2, 256, 2080, 0, 2049), (1, 256, 64, 40, 9),
    (1, 128, 32, 4, 4), (2, 256, 32, 1, 30), (3, 128, 64, 6, 50), (2, 256, 64, 19, 26)])
def test_pack_and_unpack_bitwise(gpu, kv_heads, head_dim, capacity, first, count, shift, sides):
    torch, lib = gpu, library()
    rng = np.random.default_rng(first + count)
    size = kv_heads * capacity * head_dim
    rows = [rng.integers(0, 1 << 16, (count, kv_heads, head_dim), dtype=np.uint16) for _ in 'kv']
    pages = [rng.integers(0, 1 << 16, size, dtype=np.uint16) for _ in 'kv']
    want = []
    for side in range(2):
        p = pages[side].reshape(kv_heads, -1).copy()
        off = (layout.v_offsets if side else layout.k_offsets)(capacity, head_dim)[first:first + count]
        for h in range(kv_heads):
            p[h, off] = rows[side][:, h]
        want.append(p.reshape(-1))
    dr = [_offset(torch, r, shift) for r in rows]
    dp = [_offset(torch, p, shift) for p in pages]
    ptr = [ct.c_void_p(t.data_ptr() if 'kv'[i % 2] in sides else None) for i, t in enumerate(dp + dr)]
    stream = ct.c_void_p(torch.cuda.current_stream().cuda_stream)
    check(lib, lib.qv_kv_pack(*ptr, kv_heads, head_dim, capacity, first, count, stream))
    back = [_offset(torch, np.full(r.shape, 7, np.uint16), shift) for r in rows]
    bptr = [ct.c_void_p(t.data_ptr() if 'kv'[i] in sides else None) for i, t in enumerate(back)]
    check(lib, lib.qv_kv_unpack(*bptr, *ptr[:2], kv_heads, head_dim, capacity, first, count, stream))
    torch.cuda.synchronize()
    for side in range(2):
        got = dp[side].cpu().numpy().view(np.uint16)
        np.testing.assert_array_equal(got, want[side] if 'kv'[side] in sides else pages[side])
        if 'kv'[side] in sides:
            np.testing.assert_array_equal(back[side].cpu().numpy().view(np.uint16), rows[side].reshape(-1))
