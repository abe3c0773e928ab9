"""Attention on the matrix cores for every head width and storage type beside
bf16 with 64 (attention_mma.h) against the float64 oracle, at the edges of its
tiles: 32 queries or keys per wave, 128 per workgroup, streamed blocks of 32 or
64, kernel widths 32, 64, 96, 128 and 256.

Tolerances: bf16 storage rounds each result once (2^-9 at most, about 1.7e-3
in the norm), the bar is 4e-3; fp32 storage sums up to 300 terms of 2^-24 with
roundings in the scores ahead of them, the bar is 3e-6."""
import numpy as np
import pytest

from oracle import reference as ora
from tests.helpers import download, normal, stored, upload

pytestmark = pytest.mark.gpu

BAR = {"bfloat16": 4e-3, "float32": 3e-6}


@pytest.fixture(scope="module")
def lm():
    from qutai_amd.backends import amd, amd_lm

    amd.get_runtime()
    return amd_lm


def run(lm, dtype, dims, causal, layout, change=None, scale=None):
    """Device results and stored inputs as [batch][heads][time][dim] float64."""
    batch, time, heads, kv_heads, dim = dims
    counts = (heads, kv_heads, kv_heads, heads)
    host = [normal(sum(dims) + i, batch * time * n * dim) for i, n in enumerate(counts)]

    def split(x, n):
        if layout == 0:
            return x.reshape(batch, n, time, dim)
        return x.reshape(batch, time, n, dim).transpose(0, 2, 1, 3)

    if change:
        change(*(split(x, n) for x, n in zip(host, counts)))
    q, k, v, g = (upload(x, dtype) for x in host)
    out, lse = lm.attention(q, k, v, *dims, causal=causal, layout=layout, scale=scale)
    grads = lm.attention_backward(g, q, k, v, out, lse, *dims, causal=causal, layout=layout, scale=scale)
    inputs = [split(stored(x, dtype), n) for x, n in zip(host, counts)]
    results = [split(download(x).astype(np.float64), n) for x, n in zip((out, *grads), (heads, heads, kv_heads, kv_heads))]
    lse = download(lse).reshape((batch, time, heads) if layout else (batch, heads, time))
    return inputs, results, lse.transpose(0, 2, 1) if layout else lse


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("dims", [(1, 31, 2, 1, 8), (2, 32, 2, 2, 32), (1, 33, 4, 1, 40), (1, 127, 2, 1, 64),
                                  (1, 128, 2, 1, 96), (2, 129, 2, 1, 100), (1, 65, 4, 2, 128), (1, 300, 2, 1, 128),
                                  (1, 97, 2, 1, 136), (1, 160, 1, 1, 256)])
@pytest.mark.parametrize("causal,layout", [(True, 1), (False, 0), (False, 1)])
def test_edges_of_tiles_and_widths(lm, dtype, dims, causal, layout):
    (q, k, v, g), (out, dq, dk, dv), lse = run(lm, dtype, dims, causal, layout)
    batch, _, heads, kv_heads, _ = dims
    group = heads // kv_heads
    for b in range(batch):
        for kh in range(kv_heads):
            dk_sum = dv_sum = 0
            for h in range(kh * group, (kh + 1) * group):
                o_ref, l_ref = ora.attention_np(q[b, h], k[b, kh], v[b, kh], causal=causal)
                dq_ref, dk_ref, dv_ref = ora.attention_backward_np(g[b, h], q[b, h], k[b, kh], v[b, kh], o_ref, l_ref,
                                                                   causal=causal)
                dk_sum, dv_sum = dk_sum + dk_ref, dv_sum + dv_ref
                assert ora.rel_frobenius(out[b, h], o_ref) <= BAR[dtype], ("out", b, h)
                assert np.abs(lse[b, h] - l_ref).max() <= 4e-6, ("lse", b, h)  # a few ulps of the largest scores
                assert ora.rel_frobenius(dq[b, h], dq_ref) <= BAR[dtype], ("dq", b, h)
            assert ora.rel_frobenius(dk[b, kh], dk_sum) <= BAR[dtype], ("dk", b, kh)
            assert ora.rel_frobenius(dv[b, kh], dv_sum) <= BAR[dtype], ("dv", b, kh)


@pytest.mark.parametrize("dtype,dim", [("bfloat16", 128), ("float32", 64)])
def test_infinite_and_nan_operands_stay_where_they_are(lm, dtype, dim):
    """An infinity in the last value and a NaN in the last key of a causal
    sequence: every earlier query is what it is without them, bit pattern
    aside, and the last one is not finite."""
    def poison(q, k, v, g):
        v[0, 0, -1, 3] = np.inf
        k[0, 0, -2, 5] = np.nan
        q[0, 0, :, 7] = 0

    def clean(q, k, v, g):
        q[0, 0, :, 7] = 0

    dims = (1, 150, 1, 1, dim)
    (q, k, v, _), (out, dq, _, _), lse = run(lm, dtype, dims, True, 1, clean)
    _, (bad_out, bad_dq, _, bad_dv), bad_lse = run(lm, dtype, dims, True, 1, poison)
    assert ora.rel_frobenius(bad_out[0, 0, :148], out[0, 0, :148]) <= BAR[dtype]
    assert ora.rel_frobenius(bad_dq[0, 0, :148], dq[0, 0, :148]) <= BAR[dtype]
    assert np.abs(bad_lse[0, 0, :148] - lse[0, 0, :148]).max() <= 4e-6
    assert np.isnan(bad_out[0, 0, 148:]).all(axis=1).all() and np.isnan(bad_dv[0, 0]).any()


@pytest.mark.parametrize("dim", [16, 80, 128, 200])
@pytest.mark.parametrize("causal", [True, False])
def test_bf16_results_are_rounded_from_fp32(lm, dim, causal):
    """The share of results that are not float64's rounded to bf16.  An error of
    e of a value moves it across a rounding point, 2^-8 apart, in e / 2^-8 of
    the cases: fp32 probabilities and sums (up to some 2^-21) stay below 1 in
    1000, probabilities of 17 bits gave 2.3 in 1000."""
    dims = (1, 300, 4, 4, dim)
    (q, k, v, g), (out, _, dk, dv), _ = run(lm, "bfloat16", dims, causal, 1)
    wrong = lambda got, exact: np.mean(got != ora.bf16_round_array(exact.ravel()).reshape(got.shape))  # noqa: E731
    shares = []
    for h in range(4):
        o_ref, l_ref = ora.attention_np(q[0, h], k[0, h], v[0, h], causal=causal)
        grads = ora.attention_backward_np(g[0, h], q[0, h], k[0, h], v[0, h], out[0, h], l_ref, causal=causal)
        shares.append([wrong(got[0, h], exact) for got, exact in zip((out, dk, dv), (o_ref, *grads[1:]))])
    assert np.mean(shares) <= 1e-3


@pytest.mark.parametrize("dims", [(2, 5, 2, 2, 40), (1, 40, 2, 1, 128), (1, 130, 2, 1, 256)])
def test_a_query_of_one_key_has_no_gradient(lm, dims):
    """The first causal query's output is its value, so dP and delta are one sum
    and dQ is an exact zero (as float64 has it), not what two roundings leave."""
    _, (out, dq, _, _), _ = run(lm, "bfloat16", dims, True, 1)
    assert not dq[:, :, 0].any() and out[:, :, 0].any()


@pytest.mark.parametrize("dtype,dim", [("bfloat16", 32), ("bfloat16", 128), ("bfloat16", 136), ("float32", 32),
                                       ("float32", 64), ("float32", 100)])
@pytest.mark.parametrize("time", [1, 2, 3, 6, 7, 8, 9, 10, 11, 13, 14, 20, 21])
@pytest.mark.parametrize("heads", [2, 512])
def test_short_sequences(lm, dtype, dim, time, heads):
    """Both sides of the lines between one wave per row and tiles, for grids that
    fill the GPU and that do not."""
    (q, k, v, g), (out, dq, dk, dv), _ = run(lm, dtype, (1, time, heads, heads, dim), True, 1)
    for h in (0, heads - 1):
        o_ref, l_ref = ora.attention_np(q[0, h], k[0, h], v[0, h])
        grads = ora.attention_backward_np(g[0, h], q[0, h], k[0, h], v[0, h], out[0, h], l_ref)
        assert ora.rel_frobenius(out[0, h], o_ref) <= BAR[dtype]
        for got, exact in zip((dq, dk, dv), grads):
            # dq and dk of one position are a difference of equal sums
            assert np.linalg.norm(got[0, h] - exact) <= BAR[dtype] * max(np.linalg.norm(exact), np.linalg.norm(grads[2]))


def test_more_short_sequences_than_a_launch_holds_tiles(lm):
    """2^24 heads of one position: as many tiles of 256 threads are 2^32 threads,
    which no launch holds.  Each output is its value."""
    from qutai_amd.backends import amd

    batch, heads, dim = 4096, 4096, 8
    one, two = (amd.full(batch * heads * dim, x, dtype="bfloat16") for x in (1.0, 2.0))
    out, lse = lm.attention(one, one, two, batch, 1, heads, heads, dim)
    dq, dk, dv = lm.attention_backward(one, one, one, two, out, lse, batch, 1, heads, heads, dim)
    for got, value in ((out, 2.0), (dq, 0.0), (dk, 0.0), (dv, 1.0)):
        assert (np.frombuffer(got.to_array(), np.uint16) == np.float32(value).view(np.uint32) >> 16).all()


# Small magnitudes of q, k, v and dO: all bits count.  Results that are
# subnormal round to 2^-149 (fp32) and 2^-133 (bf16), half of which is allowed
# for each value beside the bar.
@pytest.mark.parametrize("dtype,dim", [("bfloat16", 32), ("bfloat16", 128), ("float32", 32), ("float32", 64),
                                       ("float32", 100)])
@pytest.mark.parametrize("sizes,scale", [((1, 1, 1e-39, 1), None), ((1, 1, 1e-33, 1), None), ((1, 1, 1, 1e-36), None),
                                         ((1, 1, 1, 1e-25), None), ((1e-36, 1e18, 1, 1), 1e17), ((1, 1, 1e-30, 1e-5), None),
                                         ((1e-36, 1e-3, 1, 1), 1e30), ((1e8, 1e9, 1, 1), 1e-17), ((1, 1, 1, 1), 1e-20)])
def test_small_operands_keep_their_bits(lm, dtype, dim, sizes, scale):
    def change(*tensors):
        for x, size in zip(tensors, sizes):
            x *= np.float32(size)

    (q, k, v, g), (out, dq, dk, dv), _ = run(lm, dtype, (1, 70, 2, 2, dim), True, 1, change, scale)
    step = 2.0 ** (-150 if dtype == "float32" else -134)
    for h in range(2):
        o_ref, l_ref = ora.attention_np(q[0, h], k[0, h], v[0, h], scale=scale)
        grads = ora.attention_backward_np(g[0, h], q[0, h], k[0, h], v[0, h], out[0, h], l_ref, scale=scale)
        for name, got, exact in zip(("out", "dq", "dk", "dv"), (out, dq, dk, dv), (o_ref, *grads)):
            allowed = BAR[dtype] * np.linalg.norm(exact) + step * exact.size ** 0.5
            assert np.linalg.norm(got[0, h] - exact) <= allowed, (name, np.linalg.norm(got[0, h] - exact), allowed)


@pytest.mark.parametrize("dtype,dim,counted", [("bfloat16", 64, True), ("bfloat16", 200, True), ("float32", 100, True),
                                               ("float32", 132, False), ("bfloat16", 36, False)])
def test_matrix_core_launches_are_counted(lm, dtype, dim, counted):
    from qutai_amd.backends import amd

    runtime = amd.get_runtime()
    before = runtime.mfma_launches
    run(lm, dtype, (1, 40, 2, 1, dim), True, 1)
    assert runtime.mfma_launches - before == (2 if counted else 0)


def test_rows_beyond_a_descriptor(lm):
    """Positions 87 MB apart: those from the 25th on of a block of 32 lie beyond
    the 2 GiB that a buffer descriptor spans.  Equal keys average the values, all
    ones; one that read as zeros would show."""
    from qutai_amd.backends import amd

    time, heads, dim = 48, 170000, 128
    ones = amd.full(time * heads * dim, 1.0, dtype="float32")
    out, _ = lm.attention(ones, ones, ones, 1, time, heads, heads, dim, causal=False)
    means = download(amd.mean(out, (time, heads * dim), 1))
    del out
    assert np.abs(means - 1).max() <= 1e-3
