"""A call that fails for want of memory leaves nothing behind: the next decode of
the same thread is launched and succeeds."""
import numpy as np
import pytest

import codag_amd as ca
from tests.gpu_helpers import rle_decode, say, single_chunk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("how", ["dev_alloc", "tune_run"])
def test_decode_after_a_failed_allocation(gpu_required, how):
    say(f"decode after a failed {how}")
    with ca.Context(0) as ctx:
        d = ctx.alloc(64)
        with pytest.raises(ca.CodagError):
            if how == "dev_alloc":
                ctx.alloc(1 << 60)
            else:
                ctx.tune_run(ca.RLEV1, d, 8, d, d, 1 << 60, 1, 16, d, reps=1)
        comp, off, ln = single_chunk(bytes([5, 1, 7]), pad=16)  # 8 values from 7 on
        st, out = rle_decode(ctx, ca.RLEV1, comp, off, ln, 1, 8)
        assert st.tolist() == [0] and out.tolist() == list(range(7, 15))
