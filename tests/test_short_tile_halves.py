"""GEMM_EXACT_SHORT's tiles for F16 and BF16 steps of many rounds: 32 x 16 past
two rounds of 32 x 32 tiles (BF16 up to K = 2,048), 32 x 32 to there and for the
other formats; and their bits there, against the VALU short-step tile."""

import numpy as np
import pytest

from charlotte_amd import matmul as mm
from charlotte_amd import synthetic
from tests.support.oracle_lib import BF16, F16, F32, Q4_0


@pytest.mark.parametrize("gtype,rows,columns,tokens,tile_tokens", [
    (F16, 8192, 1024, 64, 32), (F16, 8224, 1024, 64, 16), (F16, 6144, 4096, 100, 16), (F16, 6144, 4096, 64, 32),
    (BF16, 8192, 2048, 64, 32), (BF16, 8224, 2048, 64, 16), (BF16, 8224, 2080, 64, 32),
    (Q4_0, 8224, 1024, 64, 32), (F32, 8224, 1024, 64, 32), (F16, 8224, 1024, 16, 16), (F16, 2048, 1024, 32, 16),
])
def test_the_tile(gtype, rows, columns, tokens, tile_tokens):
    w = mm.Weight.shape(gtype, rows, columns)
    p = mm.plan_launch(mm.MatmulLaunch([mm.Member(w)], 16, [16]), tokens, mm.Target(256))
    assert p.kernel == mm.Kernel.GEMM_EXACT_SHORT and p.tile_tokens == tile_tokens


@pytest.mark.gpu
@pytest.mark.parametrize("gtype", [F16, BF16])
@pytest.mark.parametrize("rows,columns,tokens", [(8200, 64, 65), (8232, 160, 79), (6152, 1056, 97), (16392, 2048, 33)])
def test_edges_same_bits_as_the_valu_tile(gtype, rows, columns, tokens):
    from tests.support.gpu import Runner, bits_equal, first_difference

    rng = np.random.default_rng(rows + columns + tokens)
    stored = synthetic.weight(rng, int(gtype), rows, columns)
    x = synthetic.activations(rng, tokens, columns)
    p = mm.plan_launch(mm.MatmulLaunch([mm.Member(mm.Weight.shape(gtype, rows, columns))], 16, [16]), tokens)
    assert (p.kernel, p.tile_rows, p.tile_tokens) == (mm.Kernel.GEMM_EXACT_SHORT, 32, 16)
    outs = []
    for path in (mm.GemmPath.AUTO, mm.GemmPath.CANONICAL):
        ctx = mm.Context(0)
        ctx.set_gemm_path(path)
        w = mm.Weight(ctx, gtype, rows, columns, stored)
        outs.append(Runner(ctx).write(w, x, tokens))
        w.free()
        ctx.close()
    assert bits_equal(*outs), first_difference(*outs)
