"""CPU tests of the boundary: the C-ABI library loads without a GPU, exports every symbol that
include/vla_paged_attention.h declares, and reports errors the way the reference does."""
import os
import re

import pytest

from tests.conftest import ROOT


def test_library_exports_every_declared_symbol():
    from vllm_legacy_amd import _lib
    hdr = open(os.path.join(ROOT, "include", "vla_paged_attention.h")).read()
    hdr = re.sub(r"/\*.*?\*/", "", hdr, flags=re.S)
    declared = set(re.findall(r"\b(vla_[a-z0-9_]+)\s*\(", hdr))
    assert declared, "no declarations parsed"
    L = _lib.lib()
    missing = [n for n in sorted(declared) if not hasattr(L, n)]
    assert not missing, missing
    assert declared == set(_lib.EXPORTS)
    assert L.vla_abi_version() == 1


def test_status_strings_and_kv_dtype_names():
    from vllm_legacy_amd import _lib
    L = _lib.lib()
    assert L.vla_status_string(0) == b"ok"
    assert b"head size" in L.vla_status_string(1)
    assert b"block size" in L.vla_status_string(2)
    assert _lib.kv_dtype_code("auto") == 0
    assert _lib.kv_dtype_code("fp8") == 1 and _lib.kv_dtype_code("fp8_e4m3") == 1
    with pytest.raises(RuntimeError, match="Unsupported data type of kv cache"):
        _lib.kv_dtype_code("fp8_e5m2")


def test_argument_validation_without_gpu():
    # validation happens before any HIP call, so it can be exercised on a CPU-only host
    from vllm_legacy_amd import _lib
    L = _lib.lib()
    one = 0x1000  # never dereferenced: validation fails first
    rc = L.vla_paged_attention_v1(one, one, one, one, 1, 8, 8, 72, 16, 1.0, one, one, 4, 64, None,
                                  576, 9216, 1152, 0, 0, 1.0, 0, 0, 0, 64, 0, None)
    assert rc == 1  # head size
    rc = L.vla_paged_attention_v1(one, one, one, one, 1, 8, 8, 64, 4, 1.0, one, one, 4, 64, None,
                                  512, 8192, 1024, 0, 0, 1.0, 0, 0, 0, 64, 0, None)
    assert rc == 2  # block size
    rc = L.vla_paged_attention_v1(one, one, one, one, 1, 8, 3, 64, 16, 1.0, one, one, 4, 64, None,
                                  512, 8192, 1024, 0, 0, 1.0, 0, 0, 0, 64, 0, None)
    assert rc == 5  # heads not divisible
    rc = L.vla_paged_attention_v1(one, one, one, one, 1, 8, 8, 64, 16, 1.0, one, one, 4, 64, None,
                                  512, 8192, 1024, 0, 0, 1.0, 0, 0, 8, 0, 0, None)
    assert rc == 6  # blocksparse with a non-positive sparse block size
    assert L.vla_awq_gemm(one, one, one, one, one, 4, 128, 32, 128, None) == 8
    assert L.vla_gptq_gemm(one, one, one, one, None, one, 4, 64, 128, 1, 1, 8, None) == 8
    assert L.vla_swap_blocks(one, one, one, 1, 64, 9, None) == 5


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    from vllm_legacy_amd import _lib
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "nope.so"))
    with pytest.raises(ImportError, match="no fallback"):
        _lib.lib()


def test_v1_v2_selection_rules():
    """Host logic of forward_decode: the reference's rule when only query heads are known, the
    workgroup-count rule of the gfx950 kernels (no 8192-token cap) when KV heads are given."""
    from vllm_legacy_amd.attention.ops.paged_attn import PagedAttention as P
    # reference rule (paged_attn.py:120-121)
    assert P.use_v1(512, 1, 32) and P.use_v1(4096, 256, 32)
    assert not P.use_v1(4096, 16, 32) and not P.use_v1(8193, 256, 32)
    # gfx950 rule
    assert P.use_v1(512, 1, 32, 8)                 # a single partition: nothing to split
    assert not P.use_v1(4096, 8, 32, 8) and P.use_v1(4096, 16, 32, 8)
    assert P.use_v1(16384, 32, 32, 8) and not P.use_v1(16384, 8, 32, 8)
    assert not P.use_v1(4096, 64, 8, 1) and P.use_v1(4096, 128, 8, 1)   # one KV head per rank


def test_keys_up_to_which_nothing_is_shared_out():
    """The scratch question need not be asked for as many keys as _seq_ops.KV_WHOLE_KEYS."""
    from vllm_legacy_amd import _lib, _seq_ops
    L = _lib.seq_lib()
    for tokens in (1, 3, 64):
        for heads, groups in ((1, 1), (16, 1), (32, 8)):
            most = _seq_ops.KV_WHOLE_KEYS
            assert L.vla_seq_kv_attention_scratch_floats(tokens, heads, groups, 128, 128, most, _lib.BF16) == 0
            assert (L.vla_seq_kv_attention_scratch_floats(tokens, heads, groups, 128, 128, most + 1, _lib.BF16) > 0) == \
                (tokens * groups < 256)


def test_launches_without_room_for_a_chunked_recurrence():
    from vllm_legacy_amd import _lib
    L = _lib.seq_lib()
    assert L.vla_seq_gla_chunks_scratch_floats(1 << 20, 65535, 1, 16, 16, 1) > 0
    assert L.vla_seq_gla_chunks_scratch_floats(1 << 20, 65536, 1, 16, 16, 1) == 0
    assert L.vla_seq_gla_chunks_scratch_floats(64, 1, 65536, 16, 16, 1) == 0


def test_single_rows_on_latents_are_shared_out_while_workgroups_are_few():
    """Sequences stay whole (0 ranges, no scratch) up to 192 keys, up to two for each workgroup that the step has (and 512),
    and up to two for each sequence, divided by its sets of 32 heads."""
    from vllm_legacy_amd import _lib
    L = _lib.seq_lib()
    for seqs, heads, keys, whole in ((1, 16, 192, True), (1, 16, 193, False), (64, 16, 260, False), (128, 16, 256, True),
                                     (128, 16, 400, False), (256, 16, 512, True), (256, 16, 700, False), (64, 128, 400, True),
                                     (64, 128, 700, False), (512, 16, 1000, True), (512, 16, 1100, False), (2048, 32, 400, True),
                                     (4096, 16, 200, True), (64, 16, 4001, False), (512, 128, 512, True), (512, 128, 700, False),
                                     (1024, 64, 1000, True), (1024, 64, 1100, False), (65535, 128, 1 << 14, True)):
        ranges = L.vla_seq_latent_decode_ranges(seqs, keys, heads)
        assert (ranges == 0) == whole, (seqs, heads, keys, ranges)
        assert (L.vla_seq_latent_decode_scratch_floats(ranges, heads, 512) == 0) == (ranges <= 1)


def test_up_projections_at_odd_addresses_are_not_taken():
    """The kernel reads two columns at a time; the layer's own product takes any other weights."""
    import torch

    from vllm_legacy_amd import _seq_ops as ops
    flat = torch.empty(2 * 256 * 64 + 2, dtype=torch.bfloat16)
    assert ops.latent_decode_up_supported(flat[:-2].view(2, 256, 64))
    assert ops.latent_decode_up_supported(flat[2:].view(2, 256, 64))
    assert not ops.latent_decode_up_supported(flat[1:-1].view(2, 256, 64))
    assert not ops.latent_decode_up_supported(flat[:-2].view(2, 64, 256).transpose(1, 2))


@pytest.mark.parametrize("dim,vdim,rank,width", [(128, 128, 512, 576), (8, 8, 32, 32), (128, 64, 40, 48), (64, 64, 16, 32), (12, 64, 32, 32),
                                                 (64, 68, 32, 64), (64, 64, 32, 36), (64, 64, 64, 32)])
def test_what_forms_latent_keys(dim, vdim, rank, width):
    """The query says no exactly where the forming entry refuses the sizes (ahead of any use of a pointer), also where the
    prompts' kernel itself would take what another program has formed (rank 40, 16)."""
    from vllm_legacy_amd import _lib
    L = _lib.seq_lib()
    fits = dim % 8 == 0 and vdim % 8 == 0 and rank % 32 == 0 and width % 8 == 0 and width >= rank
    for dtype in (_lib.F16, _lib.BF16):
        assert bool(L.vla_seq_latent_form_supported(dim, vdim, rank, width, dtype)) == fits
    assert not L.vla_seq_latent_form_supported(dim, vdim, rank, width, _lib.F32)
    if not fits:
        assert L.vla_seq_latent_form(*[256] * 4, 1, width, 256, 256, 1, dim, vdim, rank, _lib.F16, None) != 0
        assert (rank % 32 == 0) or L.vla_seq_latent_prompt_supported(dim, 0, vdim, rank, _lib.F16)
