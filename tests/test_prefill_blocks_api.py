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


@pytest.mark.skipif(_hipcc() is None, reason="hipcc not installed")
def test_whole_fp32_stages_are_straight_line(tmp_path):
    """fp32 at head_dim 64: Q K^T of a stage whose 8 sub-tiles are all seen
    (16 MFMAs each) has no branch in it."""
    ks = kernels(device_asm("paged_prefill.hip", tmp_path), "paged_prefill_kernelILi0ELi64E")
    assert len(ks) == 2, sorted(ks)  # 2 table types
    for name, ins in ks.items():
        run = most = 0
        for i in ins:
            run = 0 if i.startswith(("s_cbranch", "s_branch")) else run + i.startswith("v_mfma")
            most = max(most, run)
        assert most >= 8 * 16, (name, most)


def test_launcher_passes_every_argument_in_order():
    """The fast-call wrapper against a stand-in for mv_paged_prefill_blocks."""
    import ctypes

    from mini_vllm.attention import _mvlaunch

    restype, argtypes = _hip.SIGNATURES["mv_paged_prefill_blocks"]
    got = []
    stand_in = ctypes.CFUNCTYPE(restype, *argtypes)(lambda *a: got.append(a) or 5)
    args = [1000 + i for i in range(len(argtypes))]
    args[argtypes.index(ctypes.c_float)] = 0.125
    real = ctypes.cast(_hip.load().mv_paged_prefill_blocks, ctypes.c_void_p).value
    try:
        _mvlaunch.bind_prefill(ctypes.cast(stand_in, ctypes.c_void_p).value)
        assert _mvlaunch.prefill(*args) == 5
        assert list(got[0]) == args
        with pytest.raises(TypeError, match="34 arguments"):
            _mvlaunch.prefill(*args[:-1])
    finally:
        _mvlaunch.bind_prefill(real)


def _work_by_loops(cached, qlens, hkv, tokens, cus, max_parts):
    """The work list's definition, unit by unit: fewer units than CUs are cut at
    multiples of 256 keys into as many parts as CUs per unit, of 512 keys or
    more."""
    items, keys = [], []
    for i, (c, q) in enumerate(zip(cached, qlens)):
        for t0 in range(0, q, tokens):
            for h in range(hkv):
                items.append((i, h, t0, min(tokens, q - t0)))
                keys.append(c + t0 + items[-1][3])
    split = max(1, min(max_parts, cus // len(keys))) if 0 < len(keys) < cus else 1
    parts = []
    for ke in keys:
        blocks = -(-ke // 256)
        n = max(1, min(split, blocks // 2))
        bounds = [p * blocks // n * 256 for p in range(n)] + [ke]
        parts.append(list(zip(bounds, bounds[1:])))
    return items, parts


@pytest.mark.parametrize("cached,qlens,hkv,tokens", [
    ([1536] * 4, [512] * 4, 2, 18), ([0], [37], 2, 18), ([3584], [512], 2, 18), ([0], [8192], 4, 36),
    ([5, 0, 700], [0, 3, 41], 8, 16), ([0, 2000, 17], [900, 1, 33], 1, 128), ([7], [0], 2, 18),
])
def test_work_list_holds_every_unit_and_part_once(cached, qlens, hkv, tokens):
    from mini_vllm.attention.paged_attention_gpu import prefill_work

    at = [5 * i + 3 for i in range(len(cached))]
    buf, seqs, work, units, most = prefill_work(at, cached, qlens, hkv, tokens, 256, 8)
    items, parts = _work_by_loops(cached, qlens, hkv, tokens, 256, 8)
    starts = [sum(qlens[:i]) for i in range(len(qlens))]
    assert seqs.tolist() == [[r, c, s, q] for r, c, s, q in zip(at, cached, starts, qlens)]
    assert seqs.data_ptr() == buf.data_ptr() and buf.numel() == 2 * seqs.numel() + work.numel()
    assert units == len(items)
    assert most == max((len(p) for p in parts), default=1)
    rows = work.tolist()
    if most == 1:
        assert sorted(map(tuple, rows)) == sorted(items)
        size = [cached[r[0]] + r[2] + r[3] for r in rows]
    else:
        got = {}
        for r in rows:
            assert r[7] >> 16 == most and (r[7] >> 8) & 0xff == len(parts[items.index(tuple(r[:4]))])
            got.setdefault((tuple(r[:4]), r[6]), {})[r[7] & 0xff] = (r[4], r[5])
        assert len({u for _, u in got}) == len(got) == units and {u for _, u in got} == set(range(units))
        for (item, _), ranges in got.items():
            want = parts[items.index(item)]
            assert [ranges[p] for p in range(len(want))] == want
        size = [r[5] - r[4] for r in rows]
    assert size == sorted(size, reverse=True)  # the most keys first


def test_work_list_errors_before_anything_is_written(lib):
    """Sizes, null pointers, lengths and a capacity that the items exceed."""
    import ctypes

    def call(cached, qlens, hkv=2, tokens=18, cus=256, parts=8, cap=4096, null=()):
        n = len(cached)
        i64 = [(ctypes.c_int64 * max(n, 1))(*x) for x in ([0] * n, cached, qlens)]
        seqs, work = (ctypes.c_int64 * (4 * n + 4))(), (ctypes.c_int32 * max(cap, 1))(*[7] * max(cap, 1))
        info = (ctypes.c_int32 * 3)()
        args = [*i64, n, hkv, tokens, cus, parts, seqs, work, cap, info]
        for k in null:
            args[k] = None
        return lib.mv_prefill_work_items(*args), list(work), list(info)

    bad = _hip.MV_ERR_INVALID_ARGUMENT
    for kw in (dict(hkv=0), dict(tokens=0), dict(cus=0), dict(parts=256), dict(cap=-1)):
        assert call([0], [5], **kw)[0] == bad, kw
    for k in (0, 1, 2, 8, 9, 11):
        assert call([0], [5], null=(k,))[0] == bad, k
    for cached, qlens in (([-1], [5]), ([0, 0], [5, -1]), ([1 << 31], [5]), ([0], [1 << 31])):
        rc, work, _ = call(cached, qlens)
        assert rc == bad and set(work) == {7}
    rc, work, _ = call([0], [18 * 300], cap=4 * 600 - 1)  # 600 units of 4 ints
    assert rc == bad and set(work) == {7}
    assert call([0], [18 * 300], cap=4 * 600)[2] == [600, 600, 1]
    assert call([4000], [18], cap=8 * 256 - 1)[0] == bad  # 2 units, cut: up to 256 items of 8 ints
    assert call([4000], [18], cap=8 * 256)[2] == [16, 2, 8]
    assert call([], [])[2] == [0, 0, 1]
