"""Both forms of the dK/dV kernel -- blocks of 256 keys, blocks of 64 keys whose waves share the walk
-- on the backward's case lists, whatever form the sizes would pick by themselves: dense, packed,
random, sink keys, hand-off, two key ranges, fp32 accumulators, tile-based addressing, the bit-for-bit
guard of the hand-kept MFMA distances.  Each test below is the one of its own file, run once per form."""
import pytest

pytestmark = pytest.mark.gpu

from test_attn_bwd_gpu import (  # noqa: E402,F401
    test_bwd_accepts_plus_inf_lse_for_empty_rows, test_bwd_dense_matches_oracle,
    test_bwd_does_not_depend_on_what_the_workspace_held, test_bwd_fp16, test_bwd_into_strided_views,
    test_bwd_packed_with_trailing_pad_rows_full_of_nan, test_bwd_varlen_matches_oracle,
    test_bwd_varlen_one_key_per_sequence)
from test_bwd_statistics_gpu import test_statistics_in_the_dq_kernel_have_the_same_bits  # noqa: E402,F401
from test_dkdv_walk_gpu import (  # noqa: E402,F401
    test_blocks_whose_waves_share_the_walk, test_packs_by_their_key_tile_table)
from test_ds_handoff_gpu import (  # noqa: E402,F401
    test_handoff_dense_matches_oracle_and_recompute, test_handoff_packed_matches_oracle,
    test_handoff_with_keys_in_two_ranges)
from test_key_ranges_gpu import (  # noqa: E402,F401
    test_two_key_ranges_equal_concatenated_keys, test_two_key_ranges_match_the_oracle)
from test_long_sequence_gpu import test_tile_based_addressing_gives_the_same_bits  # noqa: E402,F401
from test_many_sequences_gpu import test_pack_of_many_short_sequences  # noqa: E402,F401
from test_mfma_hazard_guard_gpu import (  # noqa: E402,F401
    test_inline_asm_and_builtin_mfma_builds_agree_bit_for_bit)
from test_random_shapes_gpu import test_random_case_fwd_bwd, test_random_packed_case_fwd_bwd  # noqa: E402,F401
from test_wide_accumulators_gpu import (  # noqa: E402,F401
    test_backward_into_and_onto_fp32_gradient_accumulators,
    test_packed_and_two_key_ranges_with_fp32_accumulators)


@pytest.fixture(autouse=True, params=["wide", "short"])
def form(request, monkeypatch):
    """Forces the form, and sees that the library took it in every backward of the test."""
    from ring_swa import _lib

    monkeypatch.setenv("RSWA_DKDV_FORM", request.param)
    real, seen = _lib.launch, set()

    def launch(device, entry, p, *rest):
        if entry.__name__.startswith("rswa_attn_bwd"):
            seen.add(_lib.lib().rswa_attn_bwd_dkdv_keys(p))
        return real(device, entry, p, *rest)

    monkeypatch.setattr(_lib, "launch", launch)
    yield
    assert seen <= {256 if request.param == "wide" else 64}
