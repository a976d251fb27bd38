"""A misaligned range-sum buffer is refused for every step the gate splits,
also below 32 tokens, where AUTO runs such a step in one launch that does not
use the buffer; a step that does not split ignores it."""

import numpy as np
import pytest

from tests.support.oracle_lib import Q4_0

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", ["AUTO", "EXACT_MFMA", "CANONICAL"])
@pytest.mark.parametrize("tokens", [2, 31, 32])
def test_a_misaligned_buffer_is_refused(path, tokens):
    from charlotte_amd import harness as hx
    from charlotte_amd import matmul as mm
    from charlotte_amd import synthetic

    rng = np.random.default_rng(tokens)
    rows, columns = 2048, 256
    ctx = mm.Context(0)
    ctx.set_gemm_path(mm.GemmPath[path])
    w = mm.Weight(ctx, Q4_0, rows, columns, synthetic.weight(rng, Q4_0, rows, columns))
    x = hx.Buffer.of(synthetic.activations(rng, tokens, columns))
    out, sums = hx.Buffer(4 * tokens * rows), hx.Buffer(4 * 32 * tokens * rows + 4)
    try:
        m = mm.MatmulLaunch([mm.Member(w)], x.ptr, [out.ptr])
        nbytes = 4 * 32 * tokens * rows
        mm.launch(ctx, m, tokens, mm.kAlways, sums.ptr, nbytes)
        for off in (1, 2, 3):
            with pytest.raises(mm.MatmulError) as e:
                mm.launch(ctx, m, tokens, mm.kAlways, sums.ptr + off, nbytes)
            assert e.value.status == mm.Status.INVALID_ARGUMENT and "range_sums" in str(e.value)
        mm.launch(ctx, m, tokens, mm.kNever, sums.ptr + 1, nbytes)
        hx.sync()
    finally:
        for b in (x, out, sums):
            b.free()
        w.free()
        ctx.close()
