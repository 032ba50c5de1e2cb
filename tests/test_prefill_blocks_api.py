"""Host checks of mv_paged_prefill_blocks (no GPU): work-group sizes,
workspace bytes, argument errors before any launch, and the hand-off order of
the 256-row kernels' key-split merge in the built code."""

import pytest

from mini_vllm.attention import _hip
from test_merge_order import _hipcc, check_handoff, device_asm, kernels


@pytest.fixture(scope="module")
def lib():
    return _hip.load()


def test_block_tokens(lib):
    f = lib.mv_prefill_block_tokens
    assert (f(14, 2, 64, 2, 0), f(14, 2, 64, 2, 1)) == (128 // 7, 256 // 7)
    assert (f(8, 8, 128, 1, 0), f(16, 1, 128, 1, 1)) == (128, 16)
    assert f(14, 2, 64, 0, 0) == f(14, 2, 64, 0, 1) == 16  # fp32: one size
    assert f(17, 1, 64, 2, 1) == f(14, 3, 64, 2, 0) == f(14, 2, 96, 2, 0) == 0


def test_block_workspace_bytes(lib):
    f = lib.mv_paged_prefill_blocks_workspace_bytes
    assert f(10, 4, 18, 14, 2, 64, 2) == 65536 + 10 * 4 * 18 * 7 * 66 * 4
    assert f(10, 1, 18, 14, 2, 64, 2) == f(0, 4, 18, 14, 2, 64, 2) == 0
    assert f(10, 4, 37, 14, 2, 64, 2) == f(10, 4, 0, 14, 2, 64, 2) == 0
    # the older entry point's items are of mv_prefill_tokens_per_group tokens
    assert lib.mv_paged_prefill_workspace_bytes(10, 4, 14, 2, 64, 2) == f(10, 4, 16, 14, 2, 64, 2)


@pytest.mark.parametrize("tokens", [0, -1, 37])
def test_bad_item_tokens_are_refused_on_the_host(lib, tokens):
    rc = lib.mv_paged_prefill_blocks(
        16, 896, 64, 16, 128, 64, 16, 128, 64, 16, 16, 16, 1, 1, 16, 1, 16, 1, tokens, 1, 1, 16,
        896, 64, 0.125, 14, 2, 64, 16, 4, 2, None, 0, None)
    assert rc == _hip.MV_ERR_INVALID_ARGUMENT


@pytest.mark.skipif(_hipcc() is None, reason="hipcc not installed")
def test_wide_partials_are_published_before_the_counter(tmp_path):
    ks = kernels(device_asm("paged_prefill_wide.hip", tmp_path), "paged_prefill_wide_kernel")
    assert len(ks) == 8, sorted(ks)  # 2 dtypes x 2 head dims x 2 table types
    for name, ins in ks.items():
        check_handoff(name, ins)
