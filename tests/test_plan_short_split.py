"""AUTO's plan for a step its gate would split: below 32 tokens the short-step
tile in one launch, where its 16 x 16 tiles number more than an eighth of the
compute units, and past 16 tokens where K is at most 8,192; from 32 tokens, for
fewer tiles or longer rows, and under EXACT_MFMA and CANONICAL, the split."""

import pytest

from charlotte_amd import matmul as mm

K = mm.Kernel
Q4_0 = mm.TensorType.Q4_0


@pytest.mark.parametrize("rows,tokens,path,kernel", [
    (2048, 2, mm.GemmPath.AUTO, K.GEMM_EXACT_SHORT),
    (2048, 31, mm.GemmPath.AUTO, K.GEMM_EXACT_SHORT),
    (2048, 32, mm.GemmPath.AUTO, K.GEMM_EXACT_SPLIT),
    (528, 16, mm.GemmPath.AUTO, K.GEMM_EXACT_SHORT),   # 33 tiles on 256 compute units
    (512, 16, mm.GemmPath.AUTO, K.GEMM_EXACT_SPLIT),   # 32
    (512, 17, mm.GemmPath.AUTO, K.GEMM_EXACT_SHORT),   # 64
    (2048, 16, mm.GemmPath.EXACT_MFMA, K.GEMM_EXACT_SPLIT),
    (2048, 16, mm.GemmPath.CANONICAL, K.GEMM_SPLIT),
])
def test_the_plan_of_a_step_the_gate_splits(rows, tokens, path, kernel):
    w = mm.Weight.shape(Q4_0, rows, 2048)
    m = mm.MatmulLaunch([mm.Member(w)], 16, [16])
    p = mm.plan_launch(m, tokens, mm.Target(256, path), gate=mm.kAlways, range_sums_bytes=1 << 30)
    assert p.kernel == kernel and p.launches == (1 if kernel == K.GEMM_EXACT_SHORT else 2) and p.canonical
    # without the gate, or without range sums, nothing splits
    for kw in ({"gate": mm.kNever, "range_sums_bytes": 1 << 30}, {"gate": mm.kAlways, "range_sums_bytes": 0}):
        assert mm.plan_launch(m, tokens, mm.Target(256, path), **kw).launches == 1


@pytest.mark.parametrize("columns,tokens,kernel", [
    (8192, 31, K.GEMM_EXACT_SHORT), (8224, 17, K.GEMM_EXACT_SPLIT), (14336, 16, K.GEMM_EXACT_SHORT),
    (14336, 17, K.GEMM_EXACT_SPLIT), (14336, 31, K.GEMM_EXACT_SPLIT),
])
def test_long_rows_past_sixteen_tokens_split(columns, tokens, kernel):
    w = mm.Weight.shape(Q4_0, 4096, columns)
    p = mm.plan_launch(mm.MatmulLaunch([mm.Member(w)], 16, [16]), tokens, mm.Target(256), gate=mm.kAlways,
                       range_sums_bytes=1 << 30)
    assert p.kernel == kernel
