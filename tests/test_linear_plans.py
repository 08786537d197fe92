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


@pytest.mark.parametrize("vocab,tied,once", [(100_000, False, False), (100_000, True, False), (140_000, False, True), (140_000, True, True)])
def test_products_know_whether_a_steps_weights_stay_in_the_cache_beside_the_memory(vocab, tied, once):
    """A model whose layers and head together are less than 256 MB keeps them there from step to step, whatever its embedding adds (a step looks up rows of it)."""
    import torch

    from palm_infra_amd.config import config_from_dict
    from palm_infra_amd.engine import DecoderModel
    from palm_infra_amd.weights import Weights

    spec = config_from_dict(dict(architectures=["Qwen3ForCausalLM"], vocab_size=vocab, hidden_size=1024, num_hidden_layers=2, num_attention_heads=2,
                                 num_key_value_heads=1, head_dim=64, intermediate_size=64, tie_word_embeddings=tied, rope_theta=10000.0,
                                 rms_norm_eps=1e-6, max_position_embeddings=64)).spec()
    weights = Weights({ref.key: torch.empty(ref.shape, dtype=torch.float32 if ref.role == "vector" else torch.bfloat16) for ref in spec.tensor_refs()})
    model = DecoderModel(spec, weights, torch.bfloat16, "cpu")
    layer = model.layers[1]
    products = [layer.mixer.qkv, layer.mixer.out, layer.feed_forward.gate_up, layer.feed_forward.down, model.head.linear]
    assert [p.passes_once for p in products] == [once] * 5


def test_a_launch_that_knows_no_model_goes_by_its_own_matrices():
    import torch

    from palm_infra_amd.kernels import ops
    half, more = torch.empty(128 << 20, dtype=torch.uint8), torch.empty((128 << 20) + 2, dtype=torch.uint8)
    assert not ops.passes_once(None, half, half) and ops.passes_once(None, half, more)
    assert ops.passes_once(True, half) and not ops.passes_once(False, half, more)


def test_experts_know_it_too():
    import torch

    from palm_infra_amd.parts.base import Builder
    from palm_infra_amd.parts.feedforward import RoutedExperts
    from palm_infra_amd.parts.linear import Linear

    builder, experts, one = Builder(None, torch.bfloat16, "cpu"), RoutedExperts(), Linear(torch.zeros(2, 2))
    experts.of_each = [one]
    builder.note(experts)
    builder.finish()
    assert experts.passes_once is False and one.passes_once is False
