"""What the plans of the linear products say, which is known without running them."""

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


@pytest.mark.parametrize("M,N,K,pays", [
    (17, 4096, 4096, True), (48, 1024, 2048, True), (32, 5120, 5120, True),
    (32, 2560, 4096, False), (48, 1536, 2048, False), (17, 8192, 2048, False),             # the stream does not serve what reads these rows
    (33, 5120, 4096, False), (32, 2048, 6144, False),                                      # nor so many of them; too long a walk for one block
    (16, 2560, 4096, True), (16, 4096, 12288, True), (16, 5120, 17408, False)])            # few rows: as ever
def test_which_branches_fold_the_next_norm_in(core, M, N, K, pays):
    """More than 16 rows fold only where the product that reads them applies their factor itself, and only for a reader that says so."""
    from palm_infra_amd.parts import ResidualSink

    class Takes:
        takes_prenormed = True

    assert ResidualSink(None, None, reader=Takes()).fold_pays(M, N, K) == pays
    for reader in (None, object()):
        assert ResidualSink(None, None, reader=reader).fold_pays(M, N, K) == (pays and M <= 16)
