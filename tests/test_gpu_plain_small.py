"""Tests of small collectives once more with "direct" = "0": through descriptor tables and the tile kernels, which serve every
larger buffer that is not of the team form, instead of as one launch whose descriptors ride in its arguments.  Types and
operations, operand order, ragged and unaligned buffers, in place, rank groups, and the caches behind those tables."""
import pytest

import gpu_harness as gh
import test_gpu_parity as parity
import test_gpu_random as random_cases

pytestmark = pytest.mark.gpu

for _module, _names in (
        (parity, ("test_allreduce_every_type_and_op", "test_allreduce_in_place_and_unaligned", "test_reducescatter_op_type_matrix", "test_allgather",
                  "test_rhd_allreduce_bf16", "test_special_values_follow_the_selection_rule", "test_special_values_16bit",
                  "test_fp16_sum_and_product_of_every_half_with_many_partners", "test_broadcast_reduce_scatter_rooted", "test_ring_scatter",
                  "test_order_sensitive_known_answers_on_the_gpu", "test_order_sensitive_known_answers_two_level_on_the_gpu",
                  "test_two_level_allreduce", "test_two_level_allreduce_operand_order_of_max_min", "test_two_level_reducescatter",
                  "test_two_level_reduce_to_root", "test_many_shapes_evict_cached_collectives_without_leaking", "test_collectives_recorded_into_a_callers_graph",
                  "test_sizes_that_change_from_call_to_call", "test_two_hundred_buffer_sets", "test_captured_collectives_survive_cache_wrap_and_scratch_growth",
                  "test_send_recv_and_batch")),
        (random_cases, ("test_random_allreduce", "test_random_reducescatter_allgather", "test_random_rooted",
                        "test_random_allreduce_some_ranks_in_place_and_rank_groups", "test_random_reducescatter_and_reduce_on_rank_groups"))):
    for _name in _names:
        globals()[_name] = getattr(_module, _name)


@pytest.fixture(autouse=True)
def through_tables(monkeypatch):
    init, close = gh.Group.__init__, gh.Group.close

    def checked_close(self):
        info = self.info()
        close(self)
        assert info["direct"] == 0

    monkeypatch.setattr(gh.Group, "__init__", lambda self, p, **params: init(self, p, **{"direct": 0, **params}))
    monkeypatch.setattr(gh.Group, "close", checked_close)
