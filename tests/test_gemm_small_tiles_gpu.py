"""The eight-wave 128x128 (X), 128x64 (Y) and 64x64 (Z) tiles: forced, they give
the bits of the 256x256 tile (every tile sums K in the same order), and their
copies stay inside the operands (the CPU model of the kernels' addressing: the
ring that bf16 and the fp32 MFMA read, and the 16-wide K stages, some past K, in
which the fp32 parts are read)."""
import numpy as np
import pytest

from tests import gemm_bounds_model as gm
from tests.test_gemm_tiles_gpu import _run

CASES = [(200, 130, 70, 3), (129, 40, 257, 1), (64, 72, 64, 2), (1, 300, 65, 1), (700, 320, 600, 1)]
SHAPES = {"X": (128, 128, 2, 4), "Y": (128, 64, 2, 2), "Z": (64, 64, 2, 2)}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_small_tiles_are_bit_identical(tmp_path, dtype):
    base = _run("L8D2", tmp_path / "base.npz", CASES, dtype)
    for tile in SHAPES:
        other = _run(tile, tmp_path / f"{tile}.npz", CASES, dtype)
        for key in base.files:
            assert np.array_equal(base[key], other[key]), (tile, key)


@pytest.mark.parametrize("f32", [False, True], ids=["bf16", "fp32"])
@pytest.mark.parametrize("tile", [*SHAPES, "L8D2", "S", "H", "N", "W"])
def test_copies_stay_in_bounds(f32, tile):
    rng = np.random.default_rng(7)
    table = {c.name: (c.bm, c.bn, c.wm, c.wn) for c in gm.tile_configs(f32)}
    cfg = gm.Config(tile, *SHAPES.get(tile, table.get(tile)), 16 if f32 else 64, 2)
    for m, k, n in [tuple(int(v) for v in rng.integers(1, 500, size=3)) for _ in range(3)] + [(257, 65, 129), (1, 1, 1)]:
        for ta in (False, True):
            for tb in (False, True):
                gm.plain_gemm(cfg, f32, m, k, n, 1, ta, tb, out_f32=bool(rng.integers(2)))
                if k >= 129:
                    gm.plain_gemm(cfg, f32, m, k, n, 1, ta, tb, splits=3)
