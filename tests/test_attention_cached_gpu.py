"""The one-launch attention over a key/value cache against float64 attention:
head widths on both sides of each lane count, key counts around one pass of a
workgroup, the longest cache, and the queries of a short prefill."""
import numpy as np
import pytest

from oracle import reference as ora
from qutai_amd import Tensor
from qutai_amd.backends import amd, amd_lm
from qutai_amd.nn import KVCache

pytestmark = pytest.mark.gpu

CASES = [
    # dtype, batch, heads, dim, total, length
    ("bfloat16", 2, 3, 8, 1, 1), ("bfloat16", 2, 2, 40, 64, 1), ("bfloat16", 1, 2, 64, 257, 3),
    ("bfloat16", 2, 2, 136, 65, 2), ("bfloat16", 1, 1, 256, 6000, 1), ("bfloat16", 1, 9, 64, 12000, 2), ("bfloat16", 3, 2, 128, 1030, 4),
    ("float32", 2, 2, 4, 5, 5), ("float32", 1, 3, 32, 300, 4), ("float32", 2, 1, 64, 129, 1),
    ("float32", 1, 2, 100, 1000, 7), ("float32", 1, 1, 256, 3000, 1), ("float32", 5, 2, 32, 40, 8),
]


def _draw(rng, shape, dtype):
    x = rng.standard_normal(shape).astype(np.float32)
    if dtype == "bfloat16":
        x = np.asarray(ora.bf16_round_array(x.ravel()), dtype=np.float32).reshape(shape)
    return x


@pytest.mark.parametrize("dtype,batch,heads,dim,total,length", CASES)
def test_cached_attention_matches_float64(dtype, batch, heads, dim, total, length):
    rng = np.random.default_rng(dim + total)
    q = _draw(rng, (batch, length, heads, dim), dtype)
    k, v = (_draw(rng, (batch, heads, total, dim), dtype) for _ in range(2))
    stores = [amd.storage(x.ravel().tolist(), dtype=dtype) for x in (q, k, v)]
    out = amd_lm.attention_cached(*stores, batch, length, total, heads, dim)
    assert out.dtype == dtype
    got = np.array(out.tolist()).reshape(batch, length, heads, dim)
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    eps, scale = 2.0 ** -24, dim ** -0.5
    for b in range(batch):
        for h in range(heads):
            s = q[b, :, h] @ k[b, h].T * scale
            hidden = np.arange(total)[None] > total - length + np.arange(length)[:, None]
            s[hidden] = -np.inf
            x = s - s.max(axis=1, keepdims=True)
            p = np.exp(x)
            p /= p.sum(axis=1, keepdims=True)
            expected = p @ v[b, h]
            # a score's rounding (dim terms, the scale, the subtraction) and the exponential's
            # (its argument times log2 e, two units) move each probability by `moved`, the
            # normaliser by their mean; `total` more roundings in each of the two sums
            size = np.abs(q[b, :, h]) @ np.abs(k[b, h]).T * scale
            arg = np.where(hidden, 0.0, np.abs(x))
            moved = eps * ((dim + 2) * (size + size.max(axis=1, keepdims=True)) + 3 * arg + 4)
            bound = (p * (moved + (p * moved).sum(axis=1, keepdims=True) + 2 * (total + 2) * eps)) @ np.abs(v[b, h])
            bound += 2 * eps * np.abs(expected)
            if dtype == "bfloat16":
                bound += 2.0 ** -8 * (np.abs(expected) + bound)
            assert (np.abs(got[b, :, h] - expected) <= bound).all()


def test_cached_attention_refuses_what_its_kernel_cannot_hold():
    one = amd_lm.AMDStorage(12 * 8, "float32")
    for length, total, dim in ((1, 12001, 8), (amd_lm.CACHED_LENGTH + 1, 12000, 8), (1, 12, 6), (1, 12, 260), (1, 12000, 256)):
        with pytest.raises(ValueError):
            amd_lm.attention_cached(one, one, one, 1, length, total, 1, dim)
    with pytest.raises(ValueError):
        amd_lm.attention_cached(one, one, one, 1, 1, 11, 1, 8)


@pytest.mark.parametrize("dtype,batch,heads,past,new,dim", [
    ("bfloat16", 1, 1, 1, 1, 8), ("bfloat16", 2, 3, 0, 2, 8), ("float32", 1, 2, 0, 1, 64), ("float32", 3, 5, 7, 2, 12), ("bfloat16", 2, 3, 127, 1, 64),
    ("float32", 2, 2, 1023, 2, 4), ("bfloat16", 2, 2, 300, 70, 128), ("float32", 1, 3, 5, 2, 6), ("bfloat16", 1, 2, 3, 1, 20),
])
def test_cache_update_joins_keys_and_values(dtype, batch, heads, past, new, dim):
    """An empty cache of its shape, rows of one chunk, around one and two segments of 1024 chunks, new positions
    longer than a workgroup's stride; the last two take the copies."""
    rng = np.random.default_rng(past)
    old, fresh = ([_draw(rng, (batch, heads, n, dim), dtype) for _ in range(2)] for n in (past, new))
    cache = KVCache()
    for pair in (old, fresh):
        got = cache.update(*(Tensor(amd.storage(x.ravel().tolist(), dtype=dtype), shape=x.shape) for x in pair))
    for x, a, b in zip(got, old, fresh):
        assert x.shape == (batch, heads, past + new, dim)
        assert np.array_equal(np.array(x.storage.tolist()).reshape(x.shape), np.concatenate((a, b), 2))
