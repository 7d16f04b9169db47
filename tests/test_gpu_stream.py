"""The stream kernel on small calls.  A call of few segments takes the chunk kernel, so
the decode and fused-step tests of the other modules run on that; here they run again
with the stream kernel forced from the host: every (head dim, page, G <= 8 or not)
instantiation, plain and fused, its exact path for large and non-finite values, the
bounded merge wait and the poisoned workspace, arbitrary workspace contents, and the
flags of replayed graphs."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from jacq_amd import workloads as wl
from tests import test_gpu_chunks as chunks
from tests import test_gpu_fused as fused
from tests import test_gpu_parity as parity
from tests.kivi_testlib import State, to_torch
from tests.test_gpu_parity import kivi  # noqa: F401  (fixture)

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _waves(kivi, geo, batch):
    """Wavefronts of a workgroup of the chunk kernel, 0 where the stream is taken."""
    out = (ctypes.c_int32 * 5)()
    kivi.lib().jacq_kivi_test_plan_decode(ctypes.byref(geo.c()), batch,
                                          ctypes.c_int64(geo.max_seq_len()), 0, 256, out)
    return out[0]


@pytest.fixture(autouse=True)
def stream(kivi):  # noqa: F811
    small = kivi.KiviGeometry(40, 8, 128, max_pages_per_seq=64, num_pages=64)
    assert _waves(kivi, small, 2) > 0
    kivi.lib().jacq_kivi_test_force_stream(1)
    try:
        assert _waves(kivi, small, 2) == 0
        yield
    finally:
        kivi.lib().jacq_kivi_test_force_stream(0)


test_decode = parity.test_runtime_decode_matches_twopass
test_gqa_ratios = parity.test_decode_other_gqa_ratios
test_residual_windows = parity.test_other_residual_windows_write_and_decode
test_step_writes = parity.test_runtime_step_writes_then_decode
test_pages = parity.test_page16_equals_page32
test_empty_and_clamped = parity.test_seq_len_zero_and_clamp
test_extreme_values = parity.test_decode_extreme_value_scales
test_nonfinite_values = parity.test_decode_nonfinite_values
test_workspace_contents = parity.test_caller_workspace_needs_no_initial_contents
test_graph_replays = parity.test_decode_graph_replays_match_eager
test_workspace_growth = parity.test_library_workspace_per_stream_survives_growth
test_merge_timeout = parity.test_merge_timeout_drains_and_is_reported
test_merge_timeout_poisons_replays = parity.test_merge_timeout_poisons_graph_replays
test_wave_stamps = parity.test_wave_stamps_cover_the_stream
test_fused_steps = fused.test_write_decode_steps_cross_age_outs
test_fused_all_age = fused.test_write_decode_every_sequence_ages_out
test_fused_equals_append_then_decode = fused.test_write_decode_equals_append_then_decode
test_fused_graph_replays = fused.test_write_decode_graph_replays
test_fused_geometries = fused.test_write_decode_other_geometries
test_fused_merge_timeout = fused.test_write_decode_merge_timeout_is_reported
test_fused_table_capacity = fused.test_write_decode_up_to_table_capacity
test_lengths = chunks.test_lengths_around_the_cut
test_long_among_short = chunks.test_one_long_sequence_among_short_ones


@pytest.mark.parametrize("nh,nkv,hd,page,R", [(10, 2, 128, 32, 64), (32, 2, 128, 16, 32),
                                              (14, 2, 64, 32, 64), (20, 2, 64, 16, 32)])
def test_more_than_one_window_of_sequences(nh, nkv, hd, page, R):
    """67 sequences (two windows of 64) on the instantiations that the lengths above leave
    out, of which every third ages a group out at the first step."""
    lens = [R + 31 + 32 * (i % 9) if i % 3 == 0 else 1 + (53 * i) % 400 for i in range(67)]
    chunks._check(nh, nkv, hd, page, R, lens, seed=nh)


@pytest.mark.parametrize("lens,most", [([40, 130, 3], 2), ([3000, 40, 2000], 4)])
def test_units_per_wavefront(kivi, lens, most):  # noqa: F811
    """A stream of fewer than 256 units is cut into runs of two, any other short of the
    device's wavefronts into runs of four."""
    w = wl.WORKLOADS["tinyllama"].scaled(batch=len(lens), ctx_lo=32)
    st = State(w, lens=lens, seed=6)
    st.build_oracle()
    geo = kivi.KiviGeometry(w.nh, w.nkv, w.hd, w.page, 32, w.residual, st.max_pages, st.num_pages)
    cache = kivi.PagedKiviCache.from_tensors(geo, to_torch(st))
    stamps = torch.zeros((8192, 4), dtype=torch.int64, device="cuda")
    assert kivi.lib().jacq_kivi_profile_wave_stamps(kivi._ptr(stamps), 8192) == 0
    try:
        cache.decode(torch.from_numpy(st.q).view(torch.float16).cuda(),
                     torch.from_numpy(st.lens.astype(np.int32)).cuda(),
                     torch.from_numpy(st.tables).cuda())
        torch.cuda.synchronize()
    finally:
        assert kivi.lib().jacq_kivi_profile_wave_stamps(None, 0) == 0
    assert int((stamps[:, 3] & 0xFFFFFFFF).max()) == most
