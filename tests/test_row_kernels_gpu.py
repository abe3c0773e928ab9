"""Column sums (one and several parts, 16-byte and single-element lanes) and the
bias add (16-byte and element-wise) at the edges of their blocks: 64 lanes,
four waves of eight rows, 32-row parts.  Bars: fp32 sums of up to 3000 terms in
chains of at most 24 (2^-24 each): 2e-6 of the norm; bf16 rounds once (2^-8)."""
import numpy as np
import pytest

from oracle import reference as ora
from tests.helpers import download, normal, stored, upload

pytestmark = pytest.mark.gpu

BAR = {"float32": 2e-6, "bfloat16": 4e-3, "float64": 1e-14}


@pytest.fixture(scope="module")
def amd():
    from qutai_amd.backends import amd

    amd.get_runtime()
    return amd


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float64"])
@pytest.mark.parametrize("outer,rows,cols", [(1, 1, 8), (1, 31, 256), (1, 33, 260), (1, 64, 512), (1, 65, 513),
                                             (1, 3000, 24), (3, 700, 40), (2, 129, 1001), (1, 1000, 1)])
def test_column_sums(amd, dtype, outer, rows, cols):
    x = normal(rows + cols, outer * rows * cols)
    got = download(amd.sum(upload(x, dtype), (outer, rows, cols), 1)).reshape(outer, cols)
    exact = stored(x, dtype).reshape(outer, rows, cols).sum(1)
    assert ora.rel_frobenius(got, exact) <= BAR[dtype]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float64"])
@pytest.mark.parametrize("outer,rows,cols", [(20001, 16, 4), (20001, 2, 3), (20000, 130, 2), (2000, 17, 16), (3, 300, 2),
                                             (1, 20000, 2), (4000, 64, 8), (500, 5, 100)])
def test_column_sums_of_few_columns(amd, dtype, outer, rows, cols):
    """A lane per column, with one and two parts, and shapes on both sides of
    the line to a workgroup per column block.  Chains of at most 65 terms."""
    x = normal(rows * cols, outer * rows * cols)
    got = download(amd.sum(upload(x, dtype), (outer, rows, cols), 1)).reshape(outer, cols)
    exact = stored(x, dtype).reshape(outer, rows, cols).sum(1)
    assert ora.rel_frobenius(got, exact) <= BAR[dtype]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float64"])
@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 4), (257, 24), (100, 513), (64, 1024)])
def test_bias_add(amd, dtype, rows, cols):
    x, bias = normal(rows, rows * cols), normal(cols, cols)
    got = download(amd.add_rows(upload(x, dtype), upload(bias, dtype), rows, cols)).reshape(rows, cols)
    exact = stored(x, dtype).reshape(rows, cols) + stored(bias, dtype)
    assert ora.rel_frobenius(got, exact) <= BAR[dtype]
    odd = amd.view(upload(np.concatenate([[0], x]), dtype), 1, rows * cols)  # not 16-byte aligned
    assert download(amd.add_rows(odd.copy(), upload(bias, dtype), rows, cols)).tobytes() == \
        download(amd.add_rows(odd, upload(bias, dtype), rows, cols)).tobytes()
