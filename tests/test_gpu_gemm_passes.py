"""GPU: tests of the kernels behind the passes of skn_gemm_q -- which decoders' prompts and larger products take -- on those kernels also
where the entry point's own choice is one launch (few rows, or a small matrix): the option "gemm.few" is off."""
import pytest

import test_gpu_gemm as gemm
import test_gpu_gemm_blocks as blocks
from skainet_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture
def passes(hip):
    hip.set_option("gemm.few", 0)
    yield hip
    hip.set_option("gemm.few", 1)


def test_few_rows_take_the_passes_by_option(passes):
    raw, a = synth.weight(synth.Q4_K, 64, 1024, seed=1), synth.activation_bf16((20, 1024), seed=2)
    w, x, c = passes.to_device(raw), passes.to_device(a), passes.alloc(4 * 20 * 64)
    before = passes.stat("launches")
    passes.gemm_q(synth.Q4_K, w, 64, 1024, x, 20, c)
    assert passes.stat("launches") - before >= 2


def test_superblock_scale_extremes(passes):
    gemm.test_gemm_q4k_superblock_scale_extremes(passes)


def test_several_row_tiles_and_ragged_columns(passes):
    gemm.test_gemm_q4k_several_row_tiles_and_ragged_columns(passes)


@pytest.mark.parametrize("qtype,m,n,k", [(gemm.Q8_0, 64, 128, 1024), (gemm.Q4_K, 1, 64, 256), (gemm.Q4_K, 33, 100, 768), (gemm.Q6_K, 130, 65, 512)])
def test_against_the_oracle(passes, qtype, m, n, k):
    gemm.test_gemm_vs_oracle(passes, qtype, m, n, k)


@pytest.mark.parametrize("qtype", [gemm.Q4_K, gemm.Q6_K])
def test_rows_apart(passes, qtype):
    gemm.test_gemm_extreme_rows(passes, qtype)
    gemm.test_gemm_rows_match_matvec(passes, qtype)


def test_large_activations_are_rescaled(passes):
    gemm.test_gemm_large_activations_are_rescaled(passes)


@pytest.mark.parametrize("m", [8, 40])
def test_q4k_extreme_rows(passes, m):
    gemm.test_gemm_q4k_extreme_rows_on_every_tile(passes, m, 0)


@pytest.mark.parametrize("m,n,k", [(160, 100, 1280), (40, 64, 256), (512, 64, 2048), (300, 200, 768)])
def test_q6k_full_range_of_the_block_fields(passes, m, n, k):
    gemm.test_gemm_q6k_full_range_of_the_block_fields(passes, m, n, k)


@pytest.mark.parametrize("qtype,m,n,k", [(synth.Q8_0, 33, 192, 4096), (gemm.Q4_K, 7, 192, 4096)])
def test_without_room_for_parts_k_is_undivided(passes, qtype, m, n, k):
    gemm.test_gemm_without_room_for_parts_leaves_k_undivided(passes, qtype, m, n, k, 0)


@pytest.mark.parametrize("name", ["q8_0", "q4_0", "q5_k"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (32, 64, 256), (33, 65, 512), (64, 63, 1280), (128, 130, 2816), (3, 600, 16384)])
def test_blocks_every_tile_height_and_remainder(passes, name, m, n, k):
    blocks.test_every_tile_height_and_remainder(passes, name, m, n, k)


@pytest.mark.parametrize("name", ["q8_0", "q4_0", "q5_k"])
def test_blocks_whole_range_of_fields_and_rows_far_apart(passes, name):
    blocks.test_whole_range_of_fields_and_rows_far_apart(passes, name)


@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (32, 65, 512), (31, 130, 2816), (3, 600, 16384)])
def test_blocks_q4_k_of_up_to_32_rows(passes, m, n, k):
    blocks.test_q4_k_of_up_to_32_rows(passes, m, n, k)


@pytest.mark.parametrize("name,t", [("q4_k", synth.Q4_K), ("q5_k", synth.Q5_K)])
def test_blocks_superblock_scales_far_apart(passes, name, t):
    blocks.test_superblock_scales_far_apart(passes, name, t)
