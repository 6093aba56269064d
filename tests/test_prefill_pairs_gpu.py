"""The prefill instances whose waves share rows: the 128-dim raw prefill (two
16-row tiles per wave; two wave groups over alternate pages where every
workgroup has a CU of its own) and the second pass of the two-pass precise
prefill, against the oracle at the sizes where they can go wrong: a last wave
with one row, with one tile or with all but one row; even and odd page counts
(for the second pass also one page, of which the second group has none), and
calls on both sides of each line of their dispatch; a row max that moves late
(outlier keys); negative and zero scales; bf16 pages, a flagged KV head among them (the
exact products); stale slots past the last key hold NaN.  Bounds: max-abs
2e-3, relative L2 1e-3 on the fp32 output, as for the other raw calls."""
import numpy as np
import pytest

from oracle import attention_ref as ref
from redshift_amd import attention as A
from redshift_amd.workloads import Workload, f32_to_bf16_bits, make_inputs, to_float
from tests.test_attention_gpu import assert_parity, gpu_attention
from tests.test_configs_gpu import PRECISE_REL_L2, precise_attention

pytestmark = pytest.mark.gpu


# kv_heads, group, tokens, position, on 256 CUs.  FEW: few rows or pages per
# head (192-row workgroups).  GROUPS: two wave groups, from 256 cached tokens on.
# SINGLE: more than 256 workgroups of 192 rows (one group, two workgroups a CU).
# ROUND: one round of 192-row workgroups.  LONG: several rounds, fewer of 192
# rows, on a long prefix.
FEW = [(1, 8, 7, 2), (2, 7, 7, 25), (1, 4, 13, 20), (2, 4, 33, 31), (1, 1, 159, 40)]
GROUPS = [(1, 5, 200, 700), (3, 8, 70, 900), (1, 1, 129, 256), (1, 1, 161, 263), (1, 12, 13, 260), (1, 4, 130, 330)]
SINGLE = [(8, 4, 1540, 5), (130, 1, 193, 0), (130, 1, 257, 40), (65, 2, 400, 600)]
ROUND = [(1, 1, 159, 1), (8, 4, 200, 0)]
LONG = [(129, 3, 130, 400)]


@pytest.mark.parametrize('dtype', ['f16', 'bf16'])
@pytest.mark.parametrize('kv,group,tokens,position', FEW + GROUPS + SINGLE + ROUND + LONG)
def test_pairs_against_oracle(gpu, kv, group, tokens, position, dtype):
    w = Workload('pairs', kv * group, kv, 128, tokens, position, 1 / 128 ** .5, dtype, tokens, 1.0, 0.5,
                 min(8, tokens + position), 8.0)
    q, k, v, _ = make_inputs(w)
    want = ref.gqa_attention(to_float(q, dtype), to_float(k, dtype), to_float(v, dtype), position, w.scale)
    assert_parity(gpu_attention(w, q, k, v, gpu, fill_nan=True, out_dtype=gpu.float32), want)


@pytest.mark.parametrize('scale', [-0.07, 0.0, 1e-30])
@pytest.mark.parametrize('head_dim,kv,group,tokens,position', [(128, 2, 4, 70, 333), (128, 130, 1, 193, 0),
                                                               (256, 2, 6, 70, 333)])
def test_scales_against_oracle(gpu, head_dim, kv, group, tokens, position, scale):
    w = Workload('scale', kv * group, kv, head_dim, tokens, position, scale, 'f16', 9, 1.0, 0.5)
    q, k, v, _ = make_inputs(w)
    want = ref.gqa_attention(to_float(q, 'f16'), to_float(k, 'f16'), to_float(v, 'f16'), position, scale)
    assert_parity(gpu_attention(w, q, k, v, gpu, fill_nan=True, out_dtype=gpu.float32), want)


@pytest.mark.parametrize('scale', [2.0 ** 3, 2.0 ** 13, -2.0 ** 20, 2.0 ** 60])
@pytest.mark.parametrize('kind,head_dim,kv,group,tokens,position', [
    ('f16', 128, 2, 8, 70, 333), ('bf16', 128, 2, 8, 70, 333), ('f16', 128, 130, 1, 193, 3),
    ('bf16', 128, 130, 1, 193, 3), ('f16', 128, 2, 4, 40, 60), ('f16', 256, 2, 6, 70, 333),
    ('bf16', 256, 2, 6, 40, 2000), ('precise', 128, 2, 4, 70, 333), ('precise', 256, 4, 6, 70, 1500),
    ('precise', 256, 200, 1, 150, 40)])
def test_scaled_scores_beyond_the_folded_exponents(gpu, kind, head_dim, kv, group, tokens, position, scale):
    """Scaled scores that grow along the keys, past 2^12 (where a wave stops
    folding the scale into its exponents) at the smallest scale and up to 2^74:
    small integers times a power of two, so that the scores are exact and equal
    ones have equal weights."""
    w = Workload('large', kv * group, kv, head_dim, tokens, position, scale, 'f16', 5)
    rng = np.random.default_rng(tokens)
    keys = position + tokens
    q = rng.integers(-2, 3, (tokens, kv * group, head_dim)).astype(np.float16)
    k = (rng.integers(-1, 2, (keys, kv, head_dim)) * (1 + np.arange(keys) // 32 % 32)[:, None, None]).astype(np.float16)
    v = rng.integers(-64, 65, k.shape).astype(np.float16) / 64
    want = ref.gqa_attention(q, k, v, position, scale)
    if kind == 'precise':
        got = precise_attention(w, q.astype(np.float32), k, v, gpu)
    else:
        if kind == 'bf16':
            w = Workload(**{**w.__dict__, 'dtype': 'bf16'})
            q, k, v = (f32_to_bf16_bits(x.astype(np.float32)) for x in (q, k, v))
        got = gpu_attention(w, q, k, v, gpu, out_dtype=gpu.float32)
    assert_parity(got, want)


@pytest.mark.parametrize('kv,group,tokens,position', [(2, 4, 70, 333), (130, 1, 193, 0)])
def test_flagged_head_takes_the_exact_products(gpu, kv, group, tokens, position):
    """KV head 1's values lie far above the fp16 range (2^20 times N(0,1)):
    its rows are held to the bounds relative to that magnitude."""
    w = Workload('flagged', kv * group, kv, 128, tokens, position, 1 / 16, 'bf16', 3, 1.0, 1.0)
    q, k, v, _ = make_inputs(w)
    v = to_float(v, 'bf16')
    v[:, 1] *= 2.0 ** 20
    v = f32_to_bf16_bits(np.ascontiguousarray(v, np.float32))
    want = ref.gqa_attention(to_float(q, 'bf16'), to_float(k, 'bf16'), to_float(v, 'bf16'), position, w.scale)
    got = gpu_attention(w, q, k, v, gpu, fill_nan=True, out_dtype=gpu.float32)
    head = slice(group, 2 * group)
    assert_parity(got[:, head] / 2.0 ** 20, want[:, head] / 2.0 ** 20)
    rest = [h for h in range(kv * group) if h not in range(group, 2 * group)]
    assert_parity(got[:, rest], want[:, rest])


@pytest.mark.parametrize('head_dim', [128, 256])
@pytest.mark.parametrize('tokens,position', [(129, 0), (150, 0), (177, 40), (192, 1), (161, 500)])
def test_precise_two_passes_against_oracle(gpu, head_dim, tokens, position):
    """200 KV heads of 129..192 rows: 192 rows per workgroup in two passes
    (one round of workgroups instead of two), whose second takes the earliest
    rows on two wave groups over alternate pages: padded tiles, a second
    pass over one page, two and more.  Bounds of the precise entry."""
    w = Workload('two_pass', 200, 200, head_dim, tokens, position, 1 / head_dim ** .5, 'f32', tokens, 1.0, 0.5,
                 min(8, position + tokens), 8.0)
    q, k, v, _ = make_inputs(w)
    k16, v16 = k.astype(np.float16), v.astype(np.float16)
    got = precise_attention(w, q, k16, v16, gpu)
    want = ref.gqa_attention(q, k16, v16, position, w.scale)
    assert_parity(got, want)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) <= PRECISE_REL_L2


@pytest.mark.parametrize('bad', [float('inf'), float('nan')])
@pytest.mark.parametrize('dtype', ['float16', 'bfloat16'])
@pytest.mark.parametrize('kv,group,tokens,position', [(130, 1, 193, 16), (2, 8, 70, 333), (8, 4, 1540, 12)])
def test_no_row_meets_values_past_its_own_tile(gpu, kv, group, tokens, position, dtype, bad):
    """A value that is not finite reaches a row that does not see it only
    through the 16-row tile that it shares a page walk with (its weight there
    is 0): the two tiles of a wave stop at their own last pages.  Rows whose
    tile ends before the bad key's page keep their bits (fp16), or stay within
    the 16-bit weights' rounding (2^-8 of unit-variance values, bf16: such a
    value sends its KV head to the exact products)."""
    torch, d = gpu, 128
    g = torch.Generator('cuda').manual_seed(tokens)
    keys, dtype = position + tokens, getattr(torch, dtype)
    cache = A.PagedKV(kv, d, A.round_capacity(keys), dtype)
    k, v = (torch.randn(keys, kv, d, generator=g, device='cuda').to(dtype) for _ in 'kv')
    q = torch.randn(tokens, kv * group, d, generator=g, device='cuda').to(dtype)
    cache.pack(k, v)
    want = A.attention(q, cache, position, d ** -.5).view(tokens, kv, group, d)
    row = np.arange(tokens * group)
    last = position + np.minimum(row // 16 * 16 + 15, row[-1]) // group      # the last key of the row's tile
    pages = torch.from_numpy((last // 32 + 1).reshape(tokens, group)).cuda()
    checked = 0
    for key in sorted({*range((position + 31) // 32 * 32, keys, 32), keys - 1}):
        hurt = v.clone()
        hurt[key] = bad
        cache.pack(k, hurt)
        got = A.attention(q, cache, position, d ** -.5).view(tokens, kv, group, d)
        clear = pages * 32 <= key
        checked += int(clear.sum())
        same = (got == want if dtype == torch.float16 else (got - want).abs() <= 2 ** -6).all(-1)
        assert bool(same.permute(0, 2, 1)[clear].all()), key
        # Every row that sees the key shows it.
        assert not bool(torch.isfinite(got[key - position:].float()).any())
    assert checked
