"""The 32-lane decode (gemv_ranges) with its steps in turn, against the CPU
oracle bit for bit, every format: rows read coalesced (F32 at K = 1,024, F16
and BF16 at 2,048, Q8_0 at 2,048 to 4,096, Q4_0 at 3,072) and directly (a
group fewer, and the other K); one row, an odd row past the steps of a batch,
a workgroup's several tiles; members at odd rows, gated pairs and a clip."""

import numpy as np
import pytest

from tests.support.oracle_lib import BF16, F16, F32, Q4_0, Q4_1, Q6_K, Q8_0

pytestmark = pytest.mark.gpu
THREADS = 16


@pytest.fixture(scope="module")
def run():
    from charlotte_amd import matmul as mm
    from tests.support.gpu import Runner

    c = mm.Context(0)
    yield Runner(c)
    c.close()


CASES = [(F32, 1024), (F32, 992), (F32, 2048), (F16, 2048), (F16, 1024), (F16, 3072), (BF16, 2048), (BF16, 2016),
         (Q8_0, 1024), (Q8_0, 2048), (Q8_0, 3072), (Q8_0, 4096), (Q8_0, 4064), (Q8_0, 6144), (Q4_0, 3072),
         (Q4_0, 4096), (Q4_0, 2016), (Q4_1, 2048), (Q4_1, 8192), (Q6_K, 3072), (Q6_K, 4096)]


@pytest.mark.parametrize("gtype,columns", CASES)
@pytest.mark.parametrize("rows", [1, 67, 2051, 41003])
def test_rows_of_every_remainder_are_the_oracles_bits(oracle, run, gtype, columns, rows):
    from charlotte_amd import matmul as mm
    from charlotte_amd import synthetic
    from tests.support.gpu import bits_equal, first_difference

    if rows * columns > 41003 * 3072:
        rows = 41003 * 3072 // columns | 1  # the oracle's time
    rng = np.random.default_rng(rows + columns)
    stored = synthetic.weight(rng, int(gtype), rows, columns)
    x = synthetic.activations(rng, 1, columns)
    w = run.weight(gtype, rows, columns, stored)
    assert mm.plan_launch(mm.MatmulLaunch([mm.Member(w)], 16, [16]), 1).kernel == mm.Kernel.GEMV_RANGES
    got = run.write(w, x, 1)
    w.free()
    want = oracle.matmul_f32(gtype, stored, rows, columns, x, threads=THREADS)
    assert bits_equal(got, want), first_difference(got, want)


@pytest.mark.parametrize("gtype,columns", [(F32, 1024), (BF16, 2048), (Q8_0, 2048), (Q8_0, 4096), (Q4_0, 3072)])
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
