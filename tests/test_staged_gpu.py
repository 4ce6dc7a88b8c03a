"""The staged multi-query path (csrc/prefill.hip) at the sizes of the other
modules' multi-query tests, which take the direct kernel by themselves: partial
query tiles, contexts shorter than the query block, non-causal windows, sinks
over several tiles, 32-token pages, unlinked and out-of-pool pages, non-finite
keys, a running max that rises in every tile, chunk calls; D 64 and 128."""
import pytest

from test_prefill_gpu import (  # noqa: F401
    test_nan_past_context_is_ignored, test_non_finite_key_outside_window_is_ignored,
    test_prefill_fp16_vs_oracle, test_prefill_int4_pages_vs_composition_oracle,
    test_prefill_out_of_pool_pages_are_skipped, test_prefill_running_max_raised_every_tile,
    test_reference_math_equivalence_multi_query)
from test_runtime_gpu import (  # noqa: F401
    test_autochunk_matches_one_shot_prefill, test_chunk_call_workspace_is_bounded_by_the_window)
from test_sweep_gpu import test_prefill_fp16_pool_sweep, test_prefill_sweep, test_small_q_len_sweep  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _staged(multi_query_path):
    multi_query_path("staged")
