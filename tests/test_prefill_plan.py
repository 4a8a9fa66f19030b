"""Tile plans of the prompt kernel (host only)."""
import pytest


@pytest.mark.parametrize("lens_q,lens_k", [([64], [2**32 + 64]), ([1], [2**31]), ([5, 64], [5, 2**31 + 7]), ([2**30, 2**30], None)])
def test_lengths_beyond_32_bits_are_refused(sb, lens_q, lens_k):
    """The kernel reads 32-bit lengths; a wrapped one would be another length (or a negative one)."""
    with pytest.raises(RuntimeError, match="without overflow"):
        sb.ops.PrefillPlan(lens_q, lens_k, "cpu")


def test_longest_length_that_fits(sb):
    plan = sb.ops.PrefillPlan([1], [2**31 - 1], "cpu")
    assert plan.seq_lens_k.tolist() == [2**31 - 1] and plan.max_k == 2**31 - 1
