"""GEMM_EXACT at its tile's edges, against the 128-row VALU tile bit for bit:
members that end inside a 32-row block, outputs no 16-byte store can take (an
odd out_width, a first output row off by one), rows and tokens one short of
and one past a tile, both token widths, every format, K of odd group counts."""

import numpy as np
import pytest

from tests.support.oracle_lib import BF16, F16, F32, Q4_0, Q4_1, Q6_K, Q8_0

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctxs():
    from charlotte_amd import matmul as mm

    exact, tile = mm.Context(0), mm.Context(0)
    exact.set_gemm_path(mm.GemmPath.EXACT_MFMA)
    tile.set_gemm_path(mm.GemmPath.CANONICAL)
    yield exact, tile
    exact.close()
    tile.close()


def _run(ctx, gtype, parts, columns, x, widths, offsets=None, **kw):
    from charlotte_amd import matmul as mm
    from tests.support.gpu import Runner

    ws = [mm.Weight(ctx, gtype, r, columns, s) for r, s in parts]
    offsets = offsets or [0] * len(ws)
    try:
        return Runner(ctx).product([mm.Member(w, output_row=o) for w, o in zip(ws, offsets)], x, len(x), widths, **kw)
    finally:
        for w in ws:
            w.free()


@pytest.mark.parametrize("gtype", [Q4_0, Q4_1, Q8_0, Q6_K, F32, F16, BF16])
@pytest.mark.parametrize("rows,columns,tokens", [(264, 544, 31), (504, 1056, 33), (16392, 96, 1025),
                                                 (16328, 96, 1001)])
def test_edges_same_bits_as_the_tile(ctxs, gtype, rows, columns, tokens):
    """(16,328 rows x 1,001 tokens take 64-token tiles, but in F32, the others 32.)"""
    from charlotte_amd import matmul as mm
    from charlotte_amd import synthetic
    from tests.support.gpu import bits_equal, first_difference

    rng = np.random.default_rng(rows + columns + tokens)
    stored = synthetic.weight(rng, int(gtype), rows, columns)
    x = synthetic.activations(rng, tokens, columns)
    shape = mm.MatmulLaunch([mm.Member(mm.Weight.shape(gtype, rows, columns))], 16, [16])
    p = mm.plan_launch(shape, tokens, mm.Target(256, mm.GemmPath.EXACT_MFMA))
    assert p.tile_tokens == (64 if tokens == 1001 and gtype != F32 else 32)
    got, want = (_run(c, gtype, [(rows, stored)], columns, x, [rows])[0] for c in ctxs)
    assert bits_equal(got, want), first_difference(got, want)


@pytest.mark.parametrize("epilogue", ["write", "qkv", "gated"])
@pytest.mark.parametrize("tokens", [3, 65])
def test_members_and_places_no_wide_store_takes(ctxs, epilogue, tokens):
    from charlotte_amd import matmul as mm
    from charlotte_amd import synthetic
    from tests.support.gpu import bits_equal, first_difference

    rng = np.random.default_rng(tokens)
    columns = 1024
    x = synthetic.activations(rng, tokens, columns)
    if epilogue == "gated":
        sizes, widths, offsets, kw = (301, 301), [303], None, {"epilogue": mm.Epilogue.GatedActivation, "out_width": 303}
    elif epilogue == "qkv":
        sizes, widths, offsets, kw = (33, 2, 95), [33, 2, 95], None, {"epilogue": mm.Epilogue.QKV}
    else:  # the middle member's two rows elsewhere, the last right after the first's
        sizes, widths, offsets, kw = (70, 2, 60), [141], [1, 139, 71], {"out_width": 141}
    parts = [(r, synthetic.weight(rng, Q4_0, r, columns)) for r in sizes]
    outs = [_run(c, Q4_0, parts, columns, x, widths, offsets, **kw) for c in ctxs]
    for got, want in zip(*outs):
        assert bits_equal(got, want), first_difference(got, want)
