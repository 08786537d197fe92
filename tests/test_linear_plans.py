"""What the plans of the linear kernels say about products that no machine here need run."""

import pytest


@pytest.fixture(scope="module")
def core():
    from palm_infra_amd.kernels import ops
    return ops.core()


@pytest.mark.parametrize("M,N,K,gated,served", [
    (32, 2008, 2048, 1, True), (40, 22008, 4096, 1, True), (17, 2002, 2048, 1, True),        # last strips that are not whole
    (32, 2003, 2048, 1, False), (32, 2003, 2048, 0, True),                                   # gate rows without their up rows
    (48, 10_400_000, 2048, 0, True), (48, 10_500_000, 2048, 0, False),                       # results beyond offsets of 32 bits
    (16, 4096, 4096, 0, False), (49, 4096, 4096, 0, False), (32, 4096, 4160, 0, False)])
def test_the_plan_for_17_to_48_rows_promises_what_its_launch_takes(core, M, N, K, gated, served):
    assert bool(core.palm_linear_ring_parts(M, N, K, gated, 0)) == served
    # the launch looks at the operands' places last: what it says is that they are not on 16 bytes, or that the product is not served
    assert core.palm_linear_ring(None, 8, 8, 8, 0, M, N, K, gated, 1, None, 0, 0.0, None, None, None) != 0
    said = core.palm_last_error().decode()
    assert ("16-byte aligned" if served else "not served") in said, said
