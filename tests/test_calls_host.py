"""The native way to the attention operators (csrc/calls.cpp) on the CPU: it takes nothing that is not a plain tensor on a GPU, and says so."""
import ctypes
import types

import pytest
import torch

from minivllm_amd import _build, _C


@pytest.fixture(scope="module")
def calls():
    _C.load()
    if _C.calls is None:
        pytest.skip("csrc/calls.cpp has not been built")
    return _C.calls


def test_calls_decline_what_is_not_theirs(calls):
    x, i, cache = torch.zeros(3, 2, 64), torch.zeros(3, dtype=torch.int64), torch.zeros(2, 16, 2, 64)
    cu = torch.tensor([0, 3], dtype=torch.int32)
    plan = lambda *a: pytest.fail("asked for a plan")
    for q in (x, None, 3, "x", x.half(), torch.nn.Parameter(x)):
        assert calls.store(q, x, cache, cache, i) is False
        assert calls.decode(q, cache, cache, None, None, cu[None], i, 1.0, 2, 2, 64, 16, None) is None
        assert calls.decode_int8(q, cache, cache, None, None, cu[None], i, 1.0, 2, 2, 64, 16, None) is None
        assert calls.prefill(q, x, x, cu, 1.0, 2, 2, 64, None, plan, None, 1 << 30) is None
        assert calls.prefill(q, x, x, cu, 1.0, 2, 2, 64, None, plan, None, 1 << 30, x, x, cu) is None
        assert calls.prefill_paged(q, cache, cache, cu[None], cu, cu, 1.0, 2, 2, 64, 16, 3, plan, None, 1 << 30) is None
        assert calls.window_prefill(q, q, x, cu, cu, 1.0, 0, None, x, None, None, None, 0.0, 0) is False
    assert calls.store() is False and calls.store(x) is False and calls.decode(x) is None and calls.decode_int8(x) is None and calls.prefill() is None
    assert calls.prefill_paged(x) is None and calls.window_prefill(x) is False                 # numbers of arguments
    with pytest.raises(TypeError):
        calls.bind([1])


def _loaded_again(monkeypatch):
    """The binding as it is before the library is first asked for."""
    for name in ("_lib", "calls"):
        monkeypatch.setattr(_C, name, None)


def test_a_module_that_cannot_be_imported_is_declined_every_time(calls, monkeypatch):
    import sys

    import minivllm_amd
    _loaded_again(monkeypatch)
    monkeypatch.setitem(sys.modules, "minivllm_amd._calls", None)          # as one built for another torch or Python
    monkeypatch.delattr(minivllm_amd, "_calls")
    with pytest.warns(RuntimeWarning, match="_calls"):
        first = _C.load()
    assert first.mvllm_version() >= 1000 and _C.calls is None
    assert _C.load() is first and _C.calls is None


def test_a_module_of_another_build_is_declined(calls, monkeypatch):
    """The library's and the module's digests of the header and of calls.cpp: others, or none, and nothing is bound."""
    lib = _C.load()
    assert lib.mvllm_calls_digest().decode() == _build.calls_digest()
    names = {name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in _C.SIGNATURES}
    for text in (b"", b"another", _build.calls_digest()[:-1].encode()):
        held = ctypes.create_string_buffer(text)
        digest = ctypes.CFUNCTYPE(ctypes.c_void_p)(lambda: ctypes.addressof(held))
        assert calls.bind({**names, "mvllm_calls_digest": ctypes.cast(digest, ctypes.c_void_p).value}) is False
    del names["mvllm_calls_digest"]
    assert calls.bind(names) is False
    with pytest.warns(RuntimeWarning, match="_calls"):
        assert _C._bind_calls(types.SimpleNamespace(mvllm_calls_digest=digest)) is None
    assert _C._bind_calls(lib) is calls


def test_a_build_that_fails_leaves_the_module_that_was_there(tmp_path, monkeypatch):
    """A kernel that does not compile, or a link that fails: neither file is replaced.  A module that does not compile: the library is
    there without one."""
    here = tmp_path / "_calls.so"
    here.write_text("before")
    monkeypatch.setattr(_build, "CALLS_PATH", str(here))

    def run(**steps):
        def built(_):
            (tmp_path / "part").write_text("built")
            return str(tmp_path / "part")
        for name, step in {"_compile": lambda src, *a: src, "_link": lambda *a: None, "_build_calls": built, **steps}.items():
            monkeypatch.setattr(_build, name, step)
        return _build.build_library(verbose=False, jobs=2)

    def broken(*a):
        raise RuntimeError("broken")

    compile_calls = _build._build_calls
    for name in ("_compile", "_link"):
        with pytest.raises(RuntimeError, match="broken"):
            run(**{name: broken})
        assert here.read_text() == "before"
    assert run() == _build.LIB_PATH and here.read_text() == "built"
    monkeypatch.setenv("CXX", "false")
    with pytest.warns(RuntimeWarning, match="calls.cpp"):
        run(_build_calls=compile_calls)
    assert not here.exists()
    monkeypatch.setenv("CXX", str(tmp_path / "there is none"))
    with pytest.warns(RuntimeWarning, match="calls.cpp"):
        run(_build_calls=compile_calls)


def test_decodes_that_overlap_have_a_workspace_each(monkeypatch):
    """Another thread's decode, on a stream of its own, while the first one's kernels may still run: its partial results lie elsewhere."""
    from minivllm_amd.layers import attention
    places = []

    def kernels(*args):
        places.append((args[-3], args[-2]))
        if len(places) == 1:
            decode()
        return 0

    lib = types.SimpleNamespace(mvllm_paged_decode=kernels, mvllm_paged_decode_int8=kernels, mvllm_paged_decode_workspace_bytes=lambda *sizes: 1 << 20)
    for name, to in {"calls": None, "load": lambda: lib, "require_cuda": lambda *t: None, "current_stream_ptr": lambda d: 0}.items():
        monkeypatch.setattr(_C, name, to)
    monkeypatch.setattr(attention, "_warn_if_generic", lambda *a: None)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    q, cache, codes, scales = torch.zeros(2, 4, 64), torch.zeros(4, 16, 2, 64), torch.zeros(4, 16, 2, 64, dtype=torch.int8), torch.ones(4, 16, 2)
    tables, rest = torch.zeros(2, 2, dtype=torch.int32), (torch.tensor([20, 30]), 1.0, 4, 2, 64, 16)
    for decode in (lambda: attention.paged_attention_decode(q, cache, cache, tables, *rest),
                   lambda: attention.paged_attention_decode_int8(q, codes, codes, scales, scales, tables, *rest)):
        places.clear()
        decode()
        (first, n), (second, m) = places
        assert n >= 1 << 20 and m >= 1 << 20 and (first + n <= second or second + m <= first)
