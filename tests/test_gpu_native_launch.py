"""The native per-layer launches (csrc/py_torch.cpp) against the Python wrappers.

Every form of the per-layer calls runs three layers twice: with the native
launches, and with them off. Same bits, same pools, and the same errors where a
later layer of a step breaks a precondition; calls that are not the plain case
(views that need a copy, another device's or type's tensors, changed metadata)
take the wrapper's own path.
"""

import pytest
import torch

from benchmarks.paged_decode_workloads import WorkloadSpec, make_case
from gpu_util import DEV, bits, say, to_device
from mini_vllm.attention import _hip
from mini_vllm.attention import paged_attention_gpu as pg
from oracle.rotary_ref import RotaryTables

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def native():
    _hip.load()
    if _hip.native is None:
        pytest.fail("_mvtorch is not built")
    pg.invalidate_cached_metadata()
    yield
    pg.invalidate_cached_metadata()


class Counted:
    """_mvtorch with the outcome of every launch noted: "launched", or "python"
    where it left the call to the wrapper."""

    LAUNCHES = ("decode_write", "decode", "cache_write", "rope_write", "prefill")

    def __init__(self, module):
        self.module, self.outcomes = module, []

    def __getattr__(self, name):
        fn = getattr(self.module, name)
        if name not in self.LAUNCHES:
            return fn

        def call(*args):
            out = fn(*args)
            assert out is None or out is True or type(out) is not int, (name, out)
            self.outcomes.append((name, "python" if out is None else "launched"))
            return out

        return call


# What layers 2 and 3 of a step do, in order (the first makes the plan and the
# checks). Strided: K, and Q unless RoPE made it anew, are left to the wrapper.
OUTCOMES = {
    ("calls", False): [("cache_write", "launched"), ("decode", "launched")],
    ("calls", True): [("cache_write", "python"), ("decode", "python")],
    ("rope_calls", False): [("rope_write", "launched"), ("decode", "launched")],
    ("rope_calls", True): [("rope_write", "python"), ("decode", "launched")],
    ("write", False): [("decode_write", "launched")], ("write", True): [("decode_write", "python")],
    ("sublayer", False): [("decode_write", "launched")],
    ("sublayer", True): [("decode_write", "python")],
}


def _step(form, dtype, strided):
    spec = WorkloadSpec("native", 14, 2, 64, 16, dtype, 5, ("fixed", [1, 17, 64, 300, 33]))
    d = to_device(make_case(spec, seed=31))
    tables = RotaryTables(64, 10000.0, 512, dtype)
    cos, sin = tables.cos.to(DEV), tables.sin.to(DEV)
    pos = d.kv_len - 1
    g = torch.Generator().manual_seed(32)
    outs = []
    for _ in range(3):
        q = torch.randn(5, 14, 64, generator=g).to(dtype).to(DEV)
        kv = torch.randn(5, 2, 2, 64, generator=g).to(dtype).to(DEV)
        nk, nv = kv[:, 0], kv[:, 1]
        if strided:  # head_dim not contiguous: the wrapper copies
            q = q.transpose(1, 2).contiguous().transpose(1, 2)
            nk = nk.transpose(1, 2).contiguous().transpose(1, 2)
        kc, vc = d.key_cache.clone(), d.value_cache.clone()
        if form == "calls":
            pg.hip_cache_write(nk, nv, kc, vc, d.slot_mapping, 16)
            out = pg.hip_decode_attention(q, kc, vc, d.block_table, d.kv_len, 16)
        elif form == "rope_calls":
            q, k = pg.hip_rope_kv_cache_write(q, nk, nv, pos, cos, sin, kc, vc, d.slot_mapping, 16)
            out = pg.hip_decode_attention(q, kc, vc, d.block_table, d.kv_len, 16)
            outs.append(k)
        else:
            extra = dict(positions=pos, cos=cos, sin=sin) if form == "sublayer" else {}
            out = pg.hip_decode_attention(q, kc, vc, d.block_table, d.kv_len, 16, new_key=nk,
                                          new_value=nv, slot_mapping=d.slot_mapping, **extra)
        outs += [out, kc, vc]
    torch.cuda.synchronize()
    return outs


@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=str)
@pytest.mark.parametrize("form", ["calls", "rope_calls", "write", "sublayer"])
def test_same_bits_with_and_without(monkeypatch, form, dtype, strided):
    say("native launches", form, dtype, strided)
    counted = Counted(_hip.native)
    monkeypatch.setattr(_hip, "native", counted)
    on = _step(form, dtype, strided)
    assert counted.outcomes == 2 * OUTCOMES[form, strided]
    pg.invalidate_cached_metadata()
    monkeypatch.setattr(_hip, "native", None)
    off = _step(form, dtype, strided)
    for x, y in zip(on, off):
        assert x.shape == y.shape and x.stride() == y.stride() and x.dtype == y.dtype
        assert torch.equal(bits(x.cpu()), bits(y.cpu()))


def _layers(form):
    """A step's first layer made, then a function that calls a second one with
    some arguments replaced."""
    spec = WorkloadSpec("native", 14, 2, 64, 16, torch.bfloat16, 3, ("fixed", [5, 40, 100]))
    d = to_device(make_case(spec, seed=33))
    args = dict(query=d.query, key_cache=d.key_cache, value_cache=d.value_cache,
                block_table=d.block_table, kv_len_after=d.kv_len, block_size=16)
    if form == "write":
        args.update(new_key=d.new_key, new_value=d.new_value, slot_mapping=d.slot_mapping)
    if form == "cache":
        args = dict(key=d.new_key, value=d.new_value, key_cache=d.key_cache,
                    value_cache=d.value_cache, slot_mapping=d.slot_mapping, block_size=16)
    fn = pg.hip_cache_write if form == "cache" else pg.hip_decode_attention
    fn(**args)
    return args, lambda **kw: fn(**{**args, **kw})


@pytest.mark.parametrize("form,change", [
    ("decode", dict(query=lambda t: t.float())), ("decode", dict(query=lambda t: t[:2])),
    ("decode", dict(key_cache=lambda t: t.half())), ("decode", dict(block_size=lambda b: 32)),
    ("decode", dict(value_cache=lambda t: t[:-1])),
    ("decode", dict(key_cache=lambda t: t.transpose(0, 1).contiguous().transpose(0, 1))),
    ("write", dict(new_key=lambda t: t[:, :1])), ("write", dict(new_value=lambda t: t.half())),
    ("write", dict(query=lambda t: t[..., :32])), ("write", dict(new_key=lambda t: t.cpu())),
    ("cache", dict(key=lambda t: t[:2])), ("cache", dict(value=lambda t: t.half())),
    ("cache", dict(key=lambda t: t.cpu())), ("cache", dict(block_size=lambda b: 8)),
])
def test_later_layers_are_refused_as_before(monkeypatch, form, change):
    say("native launches refuse", form, list(change))
    for native in (_hip.native, None):
        monkeypatch.setattr(_hip, "native", native)
        pg.invalidate_cached_metadata()
        args, call = _layers(form)
        with pytest.raises(AssertionError):
            call(**{k: f(args[k]) for k, f in change.items()})


def test_launch_words_are_packed_once_per_step(monkeypatch):
    """Also where every layer is left to the wrapper; and again when the merge
    workspace that they point at was replaced by a larger one."""
    say("native launches: words packed")
    packed = []
    real = _hip.decode_words
    monkeypatch.setattr(_hip, "decode_words", lambda *a: packed.append(a) or real(*a))
    spec = WorkloadSpec("native", 14, 2, 64, 16, torch.bfloat16, 2, ("fixed", [900, 1500]))
    d = to_device(make_case(spec, seed=35))
    q = d.query.transpose(1, 2).contiguous().transpose(1, 2)

    def call():
        return pg.hip_decode_attention(q, d.key_cache, d.value_cache, d.block_table, d.kv_len, 16)

    first = call()
    for _ in range(3):
        assert torch.equal(bits(call().cpu()), bits(first.cpu()))
    assert len(packed) == 1
    ws = pg._workspace(DEV if DEV.index is not None else torch.device("cuda", 0), 1)
    pg._workspace(ws.device, ws.numel() + 1)
    for _ in range(2):
        assert torch.equal(bits(call().cpu()), bits(first.cpu()))
    assert len(packed) == 2 and packed[0][-2] != packed[1][-2]


def test_changed_metadata_is_checked_again():
    """An in-place write to the step's slots, lengths or table is seen."""
    say("native launches: changed metadata")
    args, call = _layers("cache")
    args["slot_mapping"][0] = args["key_cache"].shape[0] * 16
    with pytest.raises(IndexError):
        call()
    for name, value, error in (("kv_len_after", 0, ValueError), ("block_table", -1, IndexError)):
        args, call = _layers("decode")
        args[name][0] = value
        with pytest.raises(error):
            call()


def test_prefill_layers(monkeypatch):
    """Prefill calls of a step, in a fused QKV buffer and as copies' input."""
    say("native launches: prefill")
    g = torch.Generator().manual_seed(34)
    qkv = torch.randn(60, 18 * 64, generator=g).to(torch.bfloat16).to(DEV)
    q, k, v = (qkv[:, a * 64:b * 64].view(60, -1, 64) for a, b in ((0, 14), (14, 16), (16, 18)))
    kc = torch.randn(8, 2, 16, 64, generator=g).to(torch.bfloat16).to(DEV)
    bt = torch.arange(8, device=DEV).view(2, 4)
    outs = []
    counted = Counted(_hip.native)
    for native in (counted, None):
        monkeypatch.setattr(_hip, "native", native)
        pg.invalidate_cached_metadata()
        for x in (q, q, q.transpose(1, 2).contiguous().transpose(1, 2)):
            outs.append(pg.hip_prefill_attention(x, k, v, kc, kc, bt, [0, 1], [20, 0], [37, 23], 16))
    for x in outs[1:]:
        assert torch.equal(bits(x.cpu()), bits(outs[0].cpu()))
    assert counted.outcomes == [("prefill", x) for x in ("launched", "launched", "python")]
