"""BRLE chunks whose streams are longer than the chunks (long literals), at both sides
of the line between four waves and one: the choice, and outputs against the oracle."""
import numpy as np
import pytest

import codag_amd as ca
from tests.gpu_helpers import say
from tests.test_gpu_bytecodec import brle_container, compare
from tests.test_gpu_byte_waves import brle_stream

pytestmark = pytest.mark.gpu


def test_choice(gpu_required):
    say("brle: long literals, the choice")
    with ca.Context(0) as ctx:
        cus = ctx.info()[1]

        def one(each, n, chunk):
            return ca.lib().codag_test_byte_one(ctx.h, 0, each * n, n, chunk)

        for each, chunk in ((66048, 65536), (65536, 65536), (98304, 98304)):
            assert [one(each, n, chunk) for n in (1, 7 * cus, 7 * cus + 1)] == [0, 0, 1]
        for each, chunk in ((65535, 65536), (98305, 98304)):
            assert [one(each, n, chunk) for n in (15 * cus, 15 * cus + 1)] == [0, 1]


@pytest.mark.parametrize("more", [0, 1])
@pytest.mark.parametrize("kind", ["noise", "period"])
def test_both_sides(gpu_required, kind, more):
    say(f"brle: long literals, {kind}, {'above' if more else 'at'} the line")
    rng = np.random.default_rng(31)
    with ca.Context(0) as ctx:
        n = 7 * ctx.info()[1] + more
        some = [brle_stream(kind, 25000 + 7 * i, rng) for i in range(5)]
        data, ptr = brle_container([some[i % 5] for i in range(n)])
        chunk = 24900  # the streams' last literals overflow
        assert ca.lib().codag_test_byte_one(ctx.h, 0, len(data), n, chunk) == more
        compare(ctx, False, data, ptr, chunk, 3)
