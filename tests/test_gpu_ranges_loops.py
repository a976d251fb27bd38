"""The 32-lane decode past its first tile: products of more tiles than the GPU
holds workgroups, where a workgroup's next tile's rows load while the last
one's sums are finished (and, coalesced, its exchange stage is used again),
against the CPU oracle bit for bit on every row. 140,001 rows in 64-row tiles,
2,188 of them for at most 1,536 workgroups, and 70,001 rows of Q8_0 K = 4,096
in 256-row tiles, 274 of them for the one workgroup a CU that their 84 KB of LDS
leaves: a 4,099-row weight, a prime number that no tile divides, over and over."""

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


@pytest.mark.parametrize("gtype,columns,rows", [
    (F32, 1024, 140001), (F32, 992, 140001), (F16, 1024, 140001), (BF16, 2048, 140001), (Q8_0, 2048, 140001),
    (Q8_0, 3072, 140001), (Q8_0, 4096, 70001), (Q4_0, 3072, 140001),  # rows read coalesced, but F32 992
    (Q4_0, 992, 140001), (Q4_1, 2048, 140001), (Q8_0, 1024, 140001), (Q6_K, 768, 140000), (Q6_K, 4096, 140000),
])
def test_every_row_of_a_looping_grid(oracle, run, gtype, columns, rows):
    from charlotte_amd import matmul as mm
    from charlotte_amd import synthetic
    from tests.support.gpu import bits_equal, first_difference

    period = 4096 if gtype == Q6_K else 4099
    rng = np.random.default_rng(columns)
    part = bytes(synthetic.weight(rng, int(gtype), period, columns))
    x = synthetic.activations(rng, 1, columns)
    times = -(-rows // period)
    stored = np.frombuffer(part * times, np.uint8)[: len(part) // period * rows]
    w = run.weight(gtype, rows, columns, stored)
    p = mm.plan_launch(mm.MatmulLaunch([mm.Member(w)], 16, [16]), 1)
    assert p.kernel == mm.Kernel.GEMV_RANGES
    assert (p.tile_rows, p.tiles) == ((256, 274) if rows == 70001 else (64, 2188))
    got = run.write(w, x, 1)
    w.free()
    want = np.tile(oracle.matmul_f32(gtype, part, period, columns, x, threads=THREADS), (1, times))[:, :rows]
    assert bits_equal(got, want), first_difference(got, want)
