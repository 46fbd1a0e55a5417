"""How the kernels for runs of rows share a step out (vla_seq_kv_attention_tiles_form, vla_seq_latent_prompt_form), at sizes
where both sides were timed: one or two groups of waves to a workgroup, tiles found by their rank or by the grid."""
import pytest

ONE, TWO, RANKED, IN_ORDER = 1, 2, 4, 8


def kv(seqs, longest, rows, heads, kv_heads, keys, window=0, keep=0, chunk=0):
    from vllm_legacy_amd import _lib
    return _lib.seq_lib().vla_seq_kv_attention_tiles_form(seqs, longest, rows, heads, kv_heads, 128, (keys + 15) // 16, 16, window, keep, chunk)


@pytest.mark.parametrize("args,want", [
    # one workgroup a CU: 44 us with two groups, 52 with one; two to a CU: 103 and 114, 63 and 76, 35 and 42
    ((1, 2047, 2047, 16, 4, 2047), TWO + RANKED), ((1, 4096, 4096, 16, 4, 4096), TWO + RANKED),
    ((16, 250, 2700, 16, 4, 3200), TWO + RANKED), ((31, 1500, 2100, 16, 4, 1500), TWO + RANKED),
    # short walks: 14 us with one group, 22 with two; 14 and 19, 10 and 15, 15 and 23
    ((40, 98, 2100, 16, 4, 98), ONE + RANKED), ((61, 256, 1456, 16, 4, 256), ONE + RANKED),
    ((100, 98, 4900, 8, 1, 98), ONE + RANKED), ((61, 200, 800, 16, 4, 210), ONE + RANKED),
    ((40, 98, 2100, 16, 4, 1600, 100), ONE + RANKED), ((40, 98, 2100, 16, 4, 1600, 0, 0, 64), ONE + RANKED),
    # a chip full of workgroups: 62 and 73
    ((4, 2047, 5543, 16, 4, 2047), ONE + RANKED),
    # no search where no workgroup is empty and walks are short: 39 us and 42, 42 and 45
    ((256, 33, 256 * 33, 16, 4, 33), ONE), ((256, 64, 11000, 16, 4, 64), ONE), ((256, 64, 11000, 16, 4, 600), ONE + RANKED),
    # the same whole tiles: 26 us in order, 47 last tiles first; smaller rows: 46 and 42
    ((128, 64, 128 * 64, 16, 4, 64), ONE + IN_ORDER), ((400, 128, 400 * 128, 8, 1, 128), ONE),
    # more sequences than a wave's registers hold
    ((257, 33, 257 * 33, 16, 4, 1000), ONE), ((300, 20, 3000, 4, 1, 1000), TWO)])
def test_key_value_prompts(args, want):
    assert kv(*args) == want


def latent(rows, seqs, longest, heads, dim, rot, vdim, ranged=0):
    from vllm_legacy_amd import _lib
    return _lib.seq_lib().vla_seq_latent_prompt_form(rows, seqs, longest, heads, dim, rot, vdim, ranged)


@pytest.mark.parametrize("args,want", [
    # 152 us with two groups, 165 with one; 78 and 83, 60 and 71, 22 and 23
    ((4096, 1, 4096, 16, 128, 64, 128), TWO + RANKED), ((4096, 2, 2048, 16, 128, 64, 128), TWO + RANKED),
    ((2128, 1, 128, 16, 128, 64, 128), TWO + RANKED), ((512, 1, 512, 16, 128, 64, 128), TWO + RANKED),
    # narrow heads: 16 and 18
    ((2800, 12, 500, 4, 64, 32, 64), TWO + RANKED),
    # two to a CU: 20 us with one group, 25 with two
    ((70 * 331, 70, 100, 4, 64, 32, 64), ONE + RANKED),
    # 10 us with one group, 18 with two; 22 and 31, 31 and 42, 52 and 63, 150 and 202, 88 and 95, 12 and 14
    ((32 * 33, 32, 33, 16, 128, 64, 128), ONE), ((32 * 128, 32, 128, 16, 128, 64, 128), ONE),
    ((8 * 512, 8, 512, 16, 128, 64, 128), ONE + RANKED), ((20 * 728, 20, 128, 16, 128, 64, 128), ONE + RANKED),
    ((16 * 2256, 16, 256, 16, 128, 64, 128), ONE + RANKED), ((3 * 2024, 3, 1024, 16, 128, 64, 128), ONE + RANKED),
    ((128, 1, 128, 16, 128, 64, 128), ONE + RANKED),
    # by the grid: 67 us, 72 by rank; 98 and 101; of different lengths by rank
    ((256 * 33, 256, 33, 16, 128, 64, 128), ONE), ((128 * 128, 128, 128, 16, 128, 64, 128), ONE),
    ((128 * 100, 128, 300, 16, 128, 64, 128), ONE + RANKED), ((200 + 60 * 210, 61, 200, 16, 128, 64, 128), ONE + RANKED), ((257 * 300, 257, 300, 16, 128, 64, 128), ONE),
    # a range of one sequence's keys: its rows are not among them
    ((64, 1, 4096, 16, 128, 64, 128, 1), TWO + RANKED), ((64, 1, 128, 16, 128, 64, 128, 1), ONE + RANKED)])
def test_latent_prompts(args, want):
    assert latent(*args) == want


def test_no_step():
    assert kv(0, 5, 5, 16, 4, 64) == kv(2, 0, 5, 16, 4, 64) == kv(2, 5, 10, 16, 5, 64) == 0
    assert latent(0, 1, 1, 16, 128, 64, 128) == latent(5, 0, 1, 16, 128, 64, 128) == 0
