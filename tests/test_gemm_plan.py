"""The GEMM's tile choice (host rule, no GPU calls): which plans the GPU tests of splits,
pairs and store policies run on."""
import pytest

from ditserve_amd import _lib
from tests.helpers import EIGHT_WAVES, SKINNY, SMALL, T128X96, T128X192, T256, gemm_plan, pair_plan

if not _lib.LIB_PATH.exists():
    pytest.skip("libditk.so not built (run python -m ditserve_amd.build)", allow_module_level=True)


@pytest.mark.parametrize("shape,want", [
    ((2, 499712, 1536, "f32"), (SKINNY, 2, SMALL)), ((17, 499712, 1536, "f32"), (EIGHT_WAVES, 17, SMALL)),
    ((666, 1536, 1536), (SMALL, 666, SMALL)), ((1560, 1536, 8960), (T128X96, 1560, SMALL)),
    ((600, 768, 1536, "f32"), (SMALL, 600, SMALL)), ((8192, 1536, 96), (EIGHT_WAVES, 8192, SMALL)),
    # full rounds of 256 x 256 tiles, then the rest
    ((14336, 1536, 8960), (T256, 10752, T128X192)), ((54560, 3072, 14336), (T256, 54528, T128X96)),
    ((10792, 4608, 1536), (T256, 10752, SMALL)),
    # gated residuals at K < 3072: 256 x 256 tiles on eight waves
    ((20000, 1536, 1536, "gate_res"), (EIGHT_WAVES, 20000, SMALL)), ((20000, 1536, 1536), (T256, 20000, SMALL)),
    ((11000, 1536, 6144, "gate_res"), (T256, 10752, T128X96))])
def test_plans(shape, want):
    assert gemm_plan(*shape) == want


def test_rows_and_tiles_of_every_plan():
    """Both parts of a plan have rows, the first one whole tile rows."""
    rows_of = {SMALL: 64, 1: 256, 2: 256, 3: 256, 4: 128, 5: 128, 6: 128, 7: 128}
    for n in (8, 96, 1536, 1544, 4608, 8960):
        for k in (64, 448, 1536, 4096, 8960):
            for m in (1, 63, 64, 257, 1560, 2305, 5001, 10793, 14337, 65520):
                for epi in ("bias", "gate_res", "f32"):
                    tile, rows, rest = gemm_plan(m, n, k, epi)
                    assert 0 < rows <= m and tile in rows_of and rest in rows_of
                    assert rows == m or (epi != "f32" and tile >= 1 and rows % rows_of[tile] == 0)


def test_pairs():
    assert pair_plan(8192, 1536, 666, 1536, 1536, "gate_res") == T256   # one round of tiles
    assert pair_plan(8192, 4608, 666, 4608, 1536) == -1                 # the text tiles would add a round
    assert pair_plan(1560, 1536, 512, 3072, 1536) >= T256               # two widths
    assert pair_plan(64, 1536, 64, 1536, 1536, "f32") == -1 and pair_plan(64, 96, 64, 96, 96) == -1
    assert pair_plan(0, 96, 64, 96, 64) == -1 and pair_plan(64, 96, 0, 96, 64) == -1
