"""The buffer for a cut product's partial sums, on the CPU."""


def test_every_product_has_partial_sums_of_its_own():
    """Two products that are queued on two streams may run at the same time."""
    from picolm_amd import kernels
    first, second = (kernels.splitk_workspace("cpu") for _ in range(2))
    assert first.data_ptr() != second.data_ptr() and first.numel() == second.numel() == kernels.SPLITK_WS_FLOATS
