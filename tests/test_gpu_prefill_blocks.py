"""mv_paged_prefill_blocks' two work-group sizes against the oracle.

The 16-bit prefill runs 128 or 256 packed query rows per work group, whichever
its launch is faster with (test_prefill_width.py). Sizes here are the
edges: chunks of one token, of a work group's tokens and one more or less;
prefixes that end at, before and after a 16-key sub-tile, a 32-key tile and a
stage (64 and 128 keys); wave rows that straddle the causal diagonal; query
heads per kv head that do and do not divide the rows; output rows that are not
16-byte aligned. Tolerance: the oracle tests' (16-bit rounding of outputs and
probabilities).
"""

import pytest
import torch

from gpu_util import DEV, TOL, say
from mini_vllm.attention import _hip
from mini_vllm.attention import paged_attention_gpu as pag
from test_gpu_prefill import _case, _ref, _run

pytestmark = pytest.mark.gpu


def _both_sizes(monkeypatch, c):
    """The case's output with 128-row and with 256-row work groups."""
    outs = []
    for wide in (0, 1):
        tokens = _hip.load().mv_prefill_block_tokens(c["hq"], c["hkv"], c["d"],
                                                     _hip.MV_DTYPE[c["dtype"]], wide)
        monkeypatch.setattr(pag, "_prefill_tokens", lambda *a, t=tokens: t)
        outs.append(_run(c))
    return outs


@pytest.mark.parametrize("shape", [(14, 2, 64, 16, torch.bfloat16), (28, 4, 128, 16, torch.float16),
                                   (8, 8, 64, 1, torch.float16), (16, 1, 128, 64, torch.bfloat16),
                                   (9, 3, 128, 32, torch.bfloat16), (10, 5, 64, 8, torch.bfloat16)],
                         ids=lambda s: f"{s[0]}-{s[1]}-{s[2]}-bs{s[3]}-{s[4]}")
def test_edges_of_tiles_and_work_groups(monkeypatch, shape):
    hq, hkv, d, bs, dt = shape
    n_rep = hq // hkv
    narrow, wide = 128 // n_rep, 256 // n_rep
    cached = [0, 0, 15, 16, 31, 33, 63, 64, 127, 129, 255, 257, 0]
    qlen = [1, narrow, narrow + 1, narrow - 1 or 1, wide, wide + 1, wide - 1 or 1, 2, 65, 1, 32, 33,
            2 * wide + 3]
    say("prefill block edges", shape, cached, qlen)
    c = _case(hq, hkv, d, bs, dt, cached, qlen, seed=21, fused=True)
    ref = _ref(c)
    for out in _both_sizes(monkeypatch, c):
        assert not torch.isnan(out).any()
        err = (out - ref).abs().max().item()
        assert err <= TOL[dt], err


@pytest.mark.parametrize("d", [64, 128])
def test_wide_key_parts_and_sharp_scores(monkeypatch, d):
    """Both sizes with their keys cut into parts (one long sequence), Q x 4:
    tiles that leave the range of the softmax reference, merged across parts."""
    say("prefill block parts", d)
    c = _case(14, 2, d, 16, torch.bfloat16, [3000], [200], seed=22)
    c["q"] = (c["q"] * 4).to(torch.bfloat16).float()
    ref = _ref(c)
    for out in _both_sizes(monkeypatch, c):
        err = (out - ref).abs().max().item()
        assert err <= TOL[torch.bfloat16], err


@pytest.mark.parametrize("shape", [(14, 2, 64, torch.float16), (28, 4, 128, torch.bfloat16),
                                   (16, 1, 128, torch.float16)], ids=str)
@pytest.mark.parametrize("rows", [32, 64, 96, 128])
def test_few_rows_and_few_keys(monkeypatch, shape, rows):
    """Work groups of fewer rows (whose other waves have none), over key ranges
    that end at, before and after the first 32 keys, the only ones the second
    set of waves has no part in, and a stage."""
    hq, hkv, d, dt = shape
    say("prefill few rows", shape, rows)
    cached = [0, 0, 0, 0, 31, 31, 32, 20, 64, 96, 127, 128]
    qlen = [1, 31, 32, 33, 1, 2, 1, 9, 5, 33, 1, 2]
    c = _case(hq, hkv, d, 16, dt, cached, qlen, seed=23)
    monkeypatch.setattr(pag, "_prefill_tokens", lambda *a: rows * hkv // hq)
    out = _run(c)
    assert not torch.isnan(out).any()
    err = (out - _ref(c)).abs().max().item()
    assert err <= TOL[dt], err


@pytest.mark.parametrize("heads,cached,qlen,later,tokens", [
    ((28, 4, 128), [0], [37], [37], 4),                      # fewest rows of one round
    ((28, 4, 128), [0, 40, 300], [5, 18, 2], [7, 9, 9], 36),  # one block each: 256 rows
    ((28, 4, 128), [64] * 3, [100, 9, 50], [1, 150, 8], 4),
    ((14, 2, 64), [0, 33], [80, 41], [121, 0], 18),
], ids=str)
def test_captured_widths(heads, cached, qlen, later, tokens):
    """A captured launch, whose work list the device builds for the width fixed
    by its rows and sequences: replays with the lengths of the capture and with
    others of the same sum, eager work in between."""
    hq, hkv, d = heads
    say("prefill captured", heads, cached, qlen)
    dt, n, t = torch.bfloat16, len(qlen), sum(qlen)
    assert pag._prefill_tokens_fixed(*heads, dt, 256, t, n) == tokens
    cases = [_case(hq, hkv, d, 16, dt, cached, ql, seed=24 + i) for i, ql in enumerate((qlen, later))]
    c = cases[0]
    dev = {k: c[k].to(dt).to(DEV) for k in ("q", "k", "v", "kc", "vc")}
    bt = c["bt"].to(DEV)
    cached_d, qlen_d = torch.tensor(cached, device=DEV), torch.tensor(qlen, device=DEV)

    def run():
        return pag.hip_prefill_attention(*(dev[k] for k in ("q", "k", "v", "kc", "vc")), bt,
                                         c["rows"], cached_d, qlen_d, 16)

    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    cid = pag.last_capture_id()
    for i in (0, 1, 0, 1):
        x = cases[i]
        for k in ("q", "k", "v", "kc", "vc"):
            dev[k].copy_(x[k].to(dt))
        bt.copy_(x["bt"])
        qlen_d.copy_(torch.tensor(x["qlen"]))
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        pag.check_deferred(cid)
        err = (out[:sum(x["qlen"])].float().cpu() - _ref(x)).abs().max().item()
        assert err <= TOL[dt], (i, err)
    pag.clear_deferred(cid)


@pytest.mark.parametrize("wide", [0, 1])
def test_output_rows_not_16_byte_aligned(wide):
    """The C ABI takes any output strides: element stores give the same bits
    as the 16-byte stores."""
    hq, hkv, d, bs, t = 14, 2, 64, 16, 70
    say("prefill blocks unaligned output", wide)
    lib = _hip.load()
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(t, h, d, generator=g).to(torch.bfloat16).to(DEV) for h in (hq, hkv, hkv))
    kc = torch.zeros(4, hkv, bs, d, dtype=torch.bfloat16, device=DEV)
    tokens = lib.mv_prefill_block_tokens(hq, hkv, d, 2, wide)
    work = torch.tensor([(0, h, t0, min(tokens, t - t0)) for t0 in range(0, t, tokens)
                         for h in range(hkv)], dtype=torch.int32, device=DEV)
    seqs = torch.tensor([[0, 0, 0, t]], dtype=torch.int64, device=DEV)
    bt = torch.zeros(1, 1, dtype=torch.int64, device=DEV)
    outs = []
    for pad in (0, 1):
        out = torch.empty(t, hq, d + pad, dtype=torch.bfloat16, device=DEV)
        rc = lib.mv_paged_prefill_blocks(
            q.data_ptr(), *q.stride()[:2], k.data_ptr(), *k.stride()[:2], v.data_ptr(),
            *v.stride()[:2], kc.data_ptr(), kc.data_ptr(), bt.data_ptr(), 1, 1, seqs.data_ptr(), 1,
            work.data_ptr(), work.shape[0], tokens, work.shape[0], 1, out.data_ptr(),
            *out.stride()[:2], d ** -0.5, hq, hkv, d, bs, 4, 2, None, 0,
            torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        torch.cuda.synchronize()
        outs.append(out[..., :d].clone())
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("dtype", [torch.int64, torch.int32], ids=str)
@pytest.mark.parametrize("where", ["device", "host"])
def test_prefix_entries_are_checked_on_the_device(monkeypatch, dtype, where):
    """The plan's table check against its definition on the host: rows and
    prefixes outside the table, entries at the pool's edges, entries past the
    prefix that do not count; tables of either type, on either side."""
    say("prefill prefix check", dtype, where)
    monkeypatch.setattr(pag, "PREFILL_HOST_CHECK_SEQS", 0)
    hq, hkv, d, bs, nb = 14, 2, 64, 16, 40
    good = torch.arange(2 * 6).view(2, 6)
    cases = [(good, [0, 1], [96, 5], True), (good, [1, 0], [0, 81], True),
             (good, [0, 2], [16, 0], False), (good, [0, -1], [16, 0], False),
             (good, [0, 1], [97, 0], False)]
    for at, ok in ((4, False), (5, True)):  # block 4 holds token 79, block 5 is past 80 tokens
        for entry in (-1, nb):
            t = good.clone()
            t[1, at] = entry
            cases.append((t, [0, 1], [16, 80], ok))
    t = torch.full((2, 600), nb - 1)  # more entries than threads
    t[0, 599] = nb
    cases += [(t, [1, 0], [9600, 9584], True), (t, [1, 0], [9600, 9585], False)]
    q = torch.zeros(2, hq, d, dtype=torch.bfloat16, device=DEV)
    k = torch.zeros(2, hkv, d, dtype=torch.bfloat16, device=DEV)
    kc = torch.zeros(nb, hkv, bs, d, dtype=torch.bfloat16, device=DEV)
    for table, rows, cached, ok in cases:
        table = table.to(dtype)
        table = table.to(DEV) if where == "device" else table
        try:
            pag._check_prefix_tables(table.cpu().long(), rows, cached, bs, nb)
            assert ok
        except IndexError:
            assert not ok
        if ok:
            pag.hip_prefill_attention(q, k, k, kc, kc, table, rows, cached, [1, 1], bs)
        else:
            with pytest.raises(IndexError, match="insufficient"):
                pag.hip_prefill_attention(q, k, k, kc, kc, table, rows, cached, [1, 1], bs)
