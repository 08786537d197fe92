"""Which of its builds the prompt attention takes for a launch, which is known without running it."""

import pytest


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("n_seqs,max_new,max_keys,nh,nkv,window,halves", [
    (1, 1, 64, 32, 8, 0, 1), (1, 320, 320, 32, 8, 0, 1), (1, 321, 321, 32, 8, 0, 2), (1, 20, 5000, 32, 8, 0, 2),        # few pages, many
    (1, 1024, 1024, 32, 8, 0, 2), (1, 1792, 1792, 32, 8, 0, 2), (1, 1793, 1793, 32, 8, 0, 1), (1, 1024, 1024, 40, 8, 0, 1),   # up to 448 blocks
    (1, 1792, 2792, 32, 8, 0, 2), (1, 1792, 3292, 32, 8, 0, 1), (1, 1100, 5000, 32, 8, 0, 1),       # a second round as long as the first
    (1, 1024, 5000, 32, 8, 0, 2), (4, 250, 250, 32, 8, 0, 1), (4, 250, 550, 32, 8, 0, 2), (4, 512, 512, 32, 8, 0, 1),
    (1, 1300, 1300, 32, 8, 64, 1), (1, 1300, 1300, 32, 8, 512, 1), (1, 1300, 1300, 32, 8, 1300, 2),  # windows: the second round is no shorter
    (1, 64, 2064, 32, 8, 64, 1), (1, 64, 2064, 32, 8, 128, 2), (1, 1000, 1000, 32, 8, 128, 1), (1, 1000, 3000, 32, 8, 2 ** 31 - 1, 2),
    (1, 300, 0, 32, 8, 0, 1), (1, 400, 0, 32, 8, 0, 2)])                                               # the keys not known: the new ones count
def test_prompt_attention_takes_halves_where_a_block_has_many_pages_to_itself(hd, n_seqs, max_new, max_keys, nh, nkv, window, halves):
    from palm_infra_amd.kernels import ops
    assert ops.attention_lib(hd).palm_attention_prefill_halves(n_seqs, max_new, max_keys, nh, nkv, window) == halves


def test_prompt_attention_of_other_head_sizes_has_no_halves():
    from palm_infra_amd.kernels import ops
    lib = ops.attention_lib(80)
    assert lib.palm_attention_prefill_halves(1, 1000, 1000, 32, 8, 0) == 1
    assert lib.palm_attention_prefill_in(None, None, None, None, None, 1, None, None, None, None, 1, 1, 1, 1, 80, 1.0, 0, 0, 1, 2, None) != 0
    assert "halves=2" in lib.palm_last_error().decode()


@pytest.mark.parametrize("starts,counts,nh,nkv,wide", [
    ([0], [13331], 32, 8, True), ([0], [3500], 32, 8, True), ([0], [2500], 32, 8, False), ([8000], [2048], 32, 8, True), ([3000], [1000], 32, 8, False),
    ([0], [4096], 16, 8, False), ([0], [8192], 16, 8, True), ([0], [4096], 16, 2, False), ([0], [8192], 8, 8, False), ([0], [13331], 8, 8, True),
    ([0], [2048], 40, 8, True), ([0], [1300], 40, 8, False), ([0], [4096], 24, 8, True),
    ([0] * 3, [3000, 1000, 100], 8, 8, False), ([0] * 3, [3000, 1000, 100], 16, 8, False), ([0] * 2, [4096] * 2, 8, 8, True), ([3000] * 6, [100] * 6, 64, 8, True)])
def test_wide_prompt_attention_is_taken_where_it_was_measured_to_be_sooner(starts, counts, nh, nkv, wide):
    from palm_infra_amd.kernels import ops
    assert ops.wide_prompt_attention(starts, counts, nh, nkv) == wide


@pytest.mark.parametrize("lengths,nh,nkv,hd,pages", [
    ([2100] + [20] * 3, 32, 8, 128, False), ([2100] + [100] * 7, 32, 8, 128, False), ([4000] + [20] * 3, 32, 8, 128, False),        # a long one beside few
    ([2100] * 2 + [100] * 6, 32, 8, 128, False), ([8000] + [100] * 7, 8, 2, 128, False), ([4000] + [400] * 7, 32, 8, 128, True),
    ([2100] + [100] * 31, 32, 8, 128, True), ([1100] + [20] * 63, 32, 8, 128, True), ([2100] * 4, 32, 8, 128, False), ([4000] * 4, 32, 8, 128, True),
    ([2049] * 8, 32, 8, 128, True), ([2500] * 8, 32, 8, 128, True), ([4000] * 8, 32, 8, 128, True), ([300] * 8, 32, 8, 128, False), ([70 + 97 * i % 1431 for i in range(45)], 32, 8, 128, True),
    ([4000] * 32 + [20] * 32, 32, 8, 128, False), ([4000, 20] * 32, 32, 8, 128, True),                    # blocks of many short sequences, or none
    ([2500] * 8, 32, 8, 64, True), ([1100] * 8, 40, 8, 128, False), ([2048] * 64, 40, 8, 128, True), ([4000], 32, 8, 128, False), ([32000], 32, 8, 128, True),
    ([1], 32, 8, 128, False), ([1] * 96, 32, 8, 128, False), ([70000] * 8, 32, 8, 80, False), ([70000] * 8, 32, 2, 128, False)])  # not served
def test_decode_attention_is_cut_by_pages_where_the_keys_that_are_there_make_it_sooner(lengths, nh, nkv, hd, pages):
    from palm_infra_amd.kernels import ops
    longest = 256
    while longest < max(lengths):
        longest *= 2
    assert ops.decode_pages_pays(lengths, nh, nkv, hd, longest) == pages


def test_a_recorded_step_is_kept_apart_by_the_attention_that_its_lengths_choose():
    import torch

    from palm_infra_amd.config import config_from_dict
    from palm_infra_amd.engine import DecoderModel
    from palm_infra_amd.weights import Weights

    spec = config_from_dict(dict(architectures=["Qwen3ForCausalLM"], vocab_size=64, hidden_size=64, num_hidden_layers=2, num_attention_heads=32,
                                 num_key_value_heads=8, head_dim=128, intermediate_size=64, tie_word_embeddings=False, rope_theta=10000.0,
                                 rms_norm_eps=1e-6, max_position_embeddings=8192)).spec()
    weights = Weights({ref.key: torch.zeros(ref.shape, dtype=torch.float32 if ref.role == "vector" else torch.bfloat16) for ref in spec.tensor_refs()})
    model = DecoderModel(spec, weights, torch.bfloat16, "cpu")
    assert model.decode_forms([2099] * 8, 4096) == (True,)                       # one answer for the layers of one shape
    assert model.decode_forms([2099] + [19] * 7, 4096) == (False,)
    assert model.decode_forms([2099] * 97, 4096) == (False,)                      # more rows than start from the projection
    assert DecoderModel(spec, weights, torch.float32, "cpu").decode_forms([2099] * 8, 4096) == (False,)


def test_steps_beside_each_other_share_no_counters():
    """The layers of a step follow each other and share the counters of the attention cut by pages; another step may run on another stream meanwhile."""
    import torch

    from palm_infra_amd.parts import make_context
    from palm_infra_amd.parts.attention import Attention

    part = Attention.__new__(Attention)
    part.nh = 4
    one, other = (make_context([0, 1, 2], [5, 6, 7], [[1]] * 3, torch.bfloat16, "cpu") for _ in range(2))
    counters = part._arrivals(one)
    assert counters.dtype == torch.int32 and counters.numel() == 12 and not counters.any()
    assert part._arrivals(one) is counters and part._arrivals(other).data_ptr() != counters.data_ptr()


@pytest.mark.parametrize("n_seqs,max_pages,served", [(96, 174762, True), (96, 174763, False), (1, (1 << 24) - 1, True), (1, 1 << 24, False), (128, 131071, True), (128, 131072, False), (0, 4, True)])
def test_decode_attention_by_pages_says_which_tables_it_takes(n_seqs, max_pages, served):
    """What is not served is known before the launch, so that a step goes by slices instead of ending in an error."""
    from palm_infra_amd.kernels import ops
    assert ops.decode_pages_serves(n_seqs, 32, 8, 128, max_pages) == served
    lib = ops.attention_lib(128)
    # (the workspace is looked for last)
    assert lib.palm_attention_decode_pages(None, None, 0, 1, None, None, 0.0, None, None, 0, 0, 1, None, None, None, max_pages, None, None, n_seqs, 32, 8, 128, 1.0, 0,
                                           None, None, None) == (0 if n_seqs == 0 else -1)
    if n_seqs:
        assert ("a workspace and counters" if served else "not served") in lib.palm_last_error().decode()
