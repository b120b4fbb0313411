"""bench.py's stage of a kernel and key of a gridding launch (CPU only)."""

import os
import sys
import types

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


@pytest.mark.parametrize("name, stage", [
    ("void tn::(anonymous namespace)::fft_rows_kernel<512, false, false>(float2*)", "fft_fwd"),
    ("void tn::(anonymous namespace)::fft_rows_kernel<512, true, false>(float2*)", "fft_adj"),
    ("void tn::(anonymous namespace)::fft_rows_kernel<256, true, true>(float2*)", "fft_adj"),
    ("void tn::(anonymous namespace)::fft_rows_kernel<256, false, true>(float2*)", "fft_fwd"),
    ("void tn::(anonymous namespace)::grid_tiles_kernel<3, 4, 1, 1>(tn::Job const*)", "grid"),
    ("tn::(anonymous namespace)::tiles_copy_kernel(tn::Job const*)", "grid"),
    ("void tn::(anonymous namespace)::interp_staged_kernel<2, 4, false, 2>(tn::Job const*)", "interp"),
])
def test_stage_of_kernels_with_more_arguments(name, stage):
    assert bench._stage_of(bench.short_kernel_name(name)) == stage


@pytest.mark.parametrize("chunk, split, coils, key", [
    (0, 0, 16, "grid|tiles|coils=16|split=384"),
    (16, 384, 16, "grid|tiles|coils=16|split=384"),  # the same launch
    (0, 0, 40, "grid|tiles|coils=24|split=384"),     # five blocks in chunks of three
    (0, 512, 3, "grid|tiles|coils=3|split=512"),
    (8, -1, 16, "grid|tiles|coils=8|split=never"),
])
def test_keys_of_the_tile_gridding(chunk, split, coils, key):
    plan = types.SimpleNamespace(grid_mode=0, grid_chunk=chunk, grid_split=split, ndim=2,
                                 interpolator=types.SimpleNamespace(grid_mode_effective=lambda: 4))
    assert bench.variant_key(plan, "grid", coils) == key
