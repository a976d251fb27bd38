"""GEMM_EXACT_SHORT's tiles at their edges, against the VALU short-step tile
bit for bit, every format: 16 x 16 with eight waves and (K of 2,048 or more)
sixteen, 32 x 16 for steps of at most 16 tokens, 32 x 32; rows and tokens one
short of and one past a tile, ranges of no, one, two and three groups, four
groups a wave and fewer."""

import numpy as np
import pytest

from tests.support.oracle_lib import BF16, F16, F32, Q4_0, Q4_1, Q6_K, Q8_0

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctxs():
    from charlotte_amd import matmul as mm

    auto, valu = mm.Context(0), mm.Context(0)
    valu.set_gemm_path(mm.GemmPath.CANONICAL)
    yield auto, valu
    auto.close()
    valu.close()


@pytest.mark.parametrize("gtype", [Q4_0, Q4_1, Q8_0, Q6_K, F32, F16, BF16])
@pytest.mark.parametrize("rows,columns,tokens,tile", [
    (40, 544, 2, (16, 16)), (264, 2080, 17, (16, 16)), (72, 3104, 16, (16, 16)), (136, 32, 15, (16, 16)),
    (8216, 96, 5, (32, 16)), (8200, 1056, 16, (32, 16)), (8232, 160, 31, (32, 32)), (4104, 2080, 33, (32, 32)),
])
def test_edges_same_bits_as_the_valu_tile(ctxs, gtype, rows, columns, tokens, tile):
    from charlotte_amd import matmul as mm
    from charlotte_amd import synthetic
    from tests.support.gpu import Runner, bits_equal, first_difference

    rng = np.random.default_rng(rows + columns + tokens)
    stored = synthetic.weight(rng, int(gtype), rows, columns)
    x = synthetic.activations(rng, tokens, columns)
    p = mm.plan_launch(mm.MatmulLaunch([mm.Member(mm.Weight.shape(gtype, rows, columns))], 16, [16]), tokens)
    assert (p.kernel, p.tile_rows, p.tile_tokens) == (mm.Kernel.GEMM_EXACT_SHORT, *tile)
    outs = []
    for ctx in ctxs:
        w = mm.Weight(ctx, gtype, rows, columns, stored)
        outs.append(Runner(ctx).write(w, x, tokens))
        w.free()
    assert bits_equal(*outs), first_difference(*outs)
