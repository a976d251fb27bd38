"""Infinite, NaN, huge, subnormal and signed-zero values through every tile of
GEMM_EXACT_SHORT and through GEMM_EXACT, every format, against the VALU tiles: NaN
where those have NaN, every other output bit for bit. Ranges of one and two
groups, and of two and three (16 x 16 with sixteen waves); in the unquantized
formats the weights hold such values too."""

import numpy as np
import pytest

from tests.support.oracle_lib import BF16, F16, F32, Q4_0, Q4_1, Q6_K, Q8_0

pytestmark = pytest.mark.gpu
COLUMNS = 1440  # 45 groups
SIXTEEN = 2080  # 65: a wave of sixteen keeps two groups or more


@pytest.fixture(scope="module")
def ctxs():
    from charlotte_amd import matmul as mm

    auto, valu, exact = mm.Context(0), mm.Context(0), mm.Context(0)
    valu.set_gemm_path(mm.GemmPath.CANONICAL)
    exact.set_gemm_path(mm.GemmPath.EXACT_MFMA)
    yield {"AUTO": auto, "CANONICAL": valu, "EXACT_MFMA": exact}
    for c in (auto, valu, exact):
        c.close()


def _inputs(rng, tokens, columns):
    x = rng.standard_normal((tokens, columns), dtype=np.float32)
    x[0, 3], x[0, 40], x[0, 41], x[0, columns - 1] = 1e28, 1e-40, -1e-42, -0.0
    x[0, 77::97] = np.float32(-1e28)
    x[1, columns // 2] = np.inf
    x[2, 5] = np.nan
    x[3] = (x[3].astype(np.float64) * 1e-39).astype(np.float32)
    x[4, columns - 40:] = -0.0  # the last groups' inputs all -0: range sums of zero products
    x[tokens - 1, :33] = np.float32(-1e-41)
    return x


def _stored(rng, gtype, rows, columns):
    """Weights; the unquantized formats' first rows hold an infinity, a NaN, subnormals and zeros of either sign."""
    from charlotte_amd import synthetic

    stored = bytearray(synthetic.weight(rng, int(gtype), rows, columns))
    special = {F32: (np.uint32, (0x7F800000, 0x7FC00000, 0x00000001, 0x80000000, 0x807FFFFF, 0xFF800000)),
               F16: (np.uint16, (0x7C00, 0x7E00, 0x0001, 0x8000, 0x83FF, 0xFC00)),
               BF16: (np.uint16, (0x7F80, 0x7FC0, 0x0001, 0x8000, 0x807F, 0xFF80))}.get(gtype)
    if special:
        kind, values = special
        w = np.frombuffer(stored, kind).reshape(rows, columns)
        for i, v in enumerate(values):
            w[i, 7 * i + 1] = v
            w[rows - 1 - i, columns - 1 - 9 * i] = v
    return bytes(stored)


@pytest.mark.parametrize("gtype", [Q4_0, Q4_1, Q8_0, Q6_K, F32, F16, BF16])
@pytest.mark.parametrize("path,rows,columns,tokens,tile", [
    ("AUTO", 640, COLUMNS, 6, (16, 16)), ("AUTO", 640, SIXTEEN, 6, (16, 16)), ("AUTO", 12296, COLUMNS, 6, (32, 16)),
    ("AUTO", 8232, COLUMNS, 31, (32, 32)), ("EXACT_MFMA", 328, COLUMNS, 35, (256, 32)),
    ("EXACT_MFMA", 16328, 96, 1001, (256, 64)),
])
def test_special_values_as_the_valu_tiles(ctxs, gtype, path, rows, columns, tokens, tile):
    from charlotte_amd import matmul as mm
    from tests.support.gpu import Runner

    if gtype == F32 and tile == (256, 64):
        tile = (256, 32)  # F32 always by 32
    rng = np.random.default_rng(rows + columns + tokens)
    stored, x = _stored(rng, gtype, rows, columns), _inputs(rng, tokens, columns)
    m = mm.MatmulLaunch([mm.Member(mm.Weight.shape(gtype, rows, columns))], 16, [16])
    p = mm.plan_launch(m, tokens, mm.Target(256, mm.GemmPath[path]))
    assert (p.tile_rows, p.tile_tokens) == tile
    outs = []
    for name in (path, "CANONICAL"):
        w = mm.Weight(ctxs[name], gtype, rows, columns, stored)
        outs.append(Runner(ctxs[name]).write(w, x, tokens))
        w.free()
    got, want = outs
    nan = np.isnan(want)
    assert nan.any() and not nan.all() and (np.isnan(got) == nan).all(), "NaN where the VALU tile has NaN"
    assert np.isinf(want).any()
    assert (got[~nan].view(np.uint32) == want[~nan].view(np.uint32)).all()
