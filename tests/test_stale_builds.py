"""Native modules left over from an older build (no GPU): a launcher without
the newer wrappers still serves the calls it has, and a library that lacks an
entry point is refused with the rebuild command."""

import shutil
import subprocess
import types

import pytest

import mini_vllm.attention as attention
from mini_vllm.attention import _hip


@pytest.fixture
def lib():
    lib = _hip.load()
    yield lib
    _hip._bind_calls(lib)


def test_launcher_without_the_prefill_wrapper(lib, monkeypatch):
    from mini_vllm.attention import _mvlaunch

    names = ("bind", "decode_write", "decode", "cache_write", "rope_write", "plan",
             "decode_write_step", "ABI", "STEP_WORDS")
    older = types.SimpleNamespace(**{n: getattr(_mvlaunch, n) for n in names})
    monkeypatch.setattr(attention, "_mvlaunch", older)
    _hip._bind_calls(lib)
    assert _hip.decode is older.decode and _hip.cache_write is older.cache_write
    assert _hip.prefill is lib.mv_paged_prefill_blocks  # through ctypes
    assert _hip.native is None  # the native launches stand in for the whole set


def test_native_launches_are_dropped_with_their_launcher(lib, monkeypatch):
    older = types.SimpleNamespace(ABI=-1, __file__="old")
    monkeypatch.setattr(attention, "_mvlaunch", older)
    with pytest.warns(RuntimeWarning, match="built for ABI -1"):
        _hip._bind_calls(lib)
    assert _hip.native is None and _hip.launcher is None
    assert _hip.prefill is lib.mv_paged_prefill_blocks


@pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc not installed")
def test_library_without_an_entry_point(tmp_path):
    missing = "mv_paged_prefill_blocks"
    src = tmp_path / "old.c"
    src.write_text("".join(f"int {n}(void) {{ return {_hip.ABI_VERSION}; }}\n"
                           for n in _hip.SIGNATURES if n != missing))
    out = tmp_path / "libold.so"
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(out)], check=True)
    with pytest.raises(RuntimeError, match=f"no {missing}.*rebuild"):
        _hip.load(str(out))
