"""Buffers that products and states work in, on the CPU."""


def test_every_product_has_partial_sums_of_its_own():
    """Two products that are queued on two streams may run at the same time."""
    from picolm_amd import kernels
    first, second = (kernels.splitk_workspace("cpu") for _ in range(2))
    assert first.data_ptr() != second.data_ptr() and first.numel() == second.numel() == kernels.SPLITK_WS_FLOATS


def test_the_chunks_scratch_has_a_bound():
    """202 heads of 128 x 128 with the delta rule are the most whose chunks fit 4 GiB in a step of 16,384 tokens."""
    from picolm_amd.parts import recurrent

    class Buffers:
        def buffer(self, name, floats, dtype):
            return floats
    rows = lambda heads: recurrent._chunk_rows(Buffers(), heads, 128, 128, 256)
    assert rows(202) == [202 * 324] and 202 * 324 * 4 * 16384 <= 4 << 30
    assert rows(203) == []
