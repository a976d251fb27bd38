"""The 32-lane decode's unquantized rows, by every way of reading them, against
the CPU oracle bit for bit: coalesced where a lane's ranges are uneven (F32
past 20 groups, F16 and BF16 past 48 and in large products), and in the widest
even ones (F32 2,048, F16 and BF16 1,024 and 3,072), a batch at a time (large F16,
BF16 and Q8_0 products) and in turn: ranges of none and one, one and two, two
and three groups, a group past and short of whole; one row, an odd row past a
batch's steps; members at odd rows, gated pairs and a clip; and more tiles than
the grid holds workgroups."""

import numpy as np
import pytest

from tests.support.oracle_lib import BF16, F16, F32, Q8_0

pytestmark = pytest.mark.gpu
THREADS = 16


@pytest.fixture(scope="module")
def run():
    from charlotte_amd import matmul as mm
    from tests.support.gpu import Runner

    c = mm.Context(0)
    yield Runner(c)
    c.close()


CASES = [(F32, 640), (F32, 704), (F32, 992), (F16, 640), (F16, 992), (BF16, 992), (Q8_0, 960), (F32, 1056), (F32, 1504), (F32, 2016), (F32, 2048), (F16, 1024), (F16, 1056), (F16, 1856), (F16, 2016),
         (F16, 2080), (F16, 2560), (F16, 3040), (F16, 3072), (BF16, 1024), (BF16, 1504), (BF16, 2080), (BF16, 3072)]


@pytest.mark.parametrize("gtype,columns", CASES)
@pytest.mark.parametrize("rows", [1, 67, 2051, 20003, 53003])
def test_rows_of_every_remainder_are_the_oracles_bits(oracle, run, gtype, columns, rows):
    from charlotte_amd import matmul as mm
    from charlotte_amd import synthetic
    from tests.support.gpu import bits_equal, first_difference

    if rows * columns > 53003 * 1056:
        rows = 53003 * 1056 // columns | 1  # the oracle's time; 2^20 groups and more all the same
    rng = np.random.default_rng(rows + columns)
    stored = synthetic.weight(rng, int(gtype), rows, columns)
    x = synthetic.activations(rng, 1, columns)
    w = run.weight(gtype, rows, columns, stored)
    assert mm.plan_launch(mm.MatmulLaunch([mm.Member(w)], 16, [16]), 1).kernel == mm.Kernel.GEMV_RANGES
    got = run.write(w, x, 1)
    w.free()
    want = oracle.matmul_f32(gtype, stored, rows, columns, x, threads=THREADS)
    assert bits_equal(got, want), first_difference(got, want)


@pytest.mark.parametrize("gtype,columns", [(F32, 800), (F32, 1504), (F32, 2048), (F16, 1856), (F16, 2560), (BF16, 3072)])
def test_members_and_gated_pairs(oracle, run, gtype, columns):
    from charlotte_amd import matmul as mm
    from charlotte_amd import synthetic
    from tests.support.gpu import bits_equal, first_difference

    rows = 4099
    rng = np.random.default_rng(columns)
    data = [synthetic.weight(rng, int(gtype), rows, columns) for _ in range(2)]
    x = synthetic.activations(rng, 1, columns)
    ws = [run.weight(gtype, rows, columns, d) for d in data]
    clip = np.array([-0.75, 0.5, -2.0, 1.5], np.float32)
    full = [oracle.matmul_f32(gtype, d, rows, columns, x, threads=THREADS) for d in data]
    got = run.product([mm.Member(ws[0], row_offset=3, rows=1001), mm.Member(ws[1], row_offset=2050, rows=2049),
                       mm.Member(ws[0], rows=77)], x, 1, [1001, 2049, 77], epilogue=mm.Epilogue.QKV)
    for g, want in zip(got, (full[0][:, 3:1004], full[1][:, 2050:4099], full[0][:, :77])):
        assert bits_equal(g, want), first_difference(g, want)
    got = run.product([mm.Member(ws[0]), mm.Member(ws[1])], x, 1, [rows], epilogue=mm.Epilogue.GatedActivation)[0]
    want = oracle.gated(full[0], full[1], activation=0)  # SiLU
    assert bits_equal(got, want), first_difference(got, want)
    got = run.product([mm.Member(ws[0])], x, 1, [rows], clip=clip)[0]
    want = oracle.finish(oracle.matmul_f32(gtype, data[0], rows, columns, oracle.clamp(x, clip[0], clip[1]),
                                           threads=THREADS), clip=clip)
    assert bits_equal(got, want), first_difference(got, want)
    for w in ws:
        w.free()


@pytest.mark.parametrize("gtype,columns", [(F32, 800), (F32, 1056), (F16, 640), (F16, 992), (F16, 1056), (BF16, 2080), (Q8_0, 992)])
def test_a_workgroup_of_several_tiles(oracle, run, gtype, columns):
    """140,001 rows, a 4,099-row weight over and over: 64-row tiles, four and
    more for each workgroup of the at most 768 that 256 compute units hold."""
    from charlotte_amd import matmul as mm
    from charlotte_amd import synthetic
    from tests.support.gpu import bits_equal, first_difference

    rows, period = 140001, 4099
    rng = np.random.default_rng(columns)
    part = bytes(synthetic.weight(rng, int(gtype), period, columns))
    x = synthetic.activations(rng, 1, columns)
    times = -(-rows // period)
    stored = np.frombuffer(part * times, np.uint8)[: len(part) // period * rows]
    w = run.weight(gtype, rows, columns, stored)
    p = mm.plan_launch(mm.MatmulLaunch([mm.Member(w)], 16, [16]), 1)
    assert p.kernel == mm.Kernel.GEMV_RANGES and p.tiles > 2 * 768
    got = run.write(w, x, 1)
    w.free()
    want = np.tile(oracle.matmul_f32(gtype, part, period, columns, x, threads=THREADS), (1, times))[:, :rows]
    assert bits_equal(got, want), first_difference(got, want)
