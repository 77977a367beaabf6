"""The CPython callables for the C entry points: the same arguments, results, conversions and errors as the ctypes functions they stand for."""
import ctypes as C

import pytest

from nanovllm_amd import _lib


@pytest.fixture(scope="module")
def dll():
    d = _lib.lib()
    if not hasattr(d.nv_attn_decode_suggest_chunk, "otherwise"):
        pytest.skip("nv_calls is not built (no Python headers)")
    return d


def test_every_entry_point_has_one(dll):
    for d, names in ((dll, _lib.PROTOTYPES), (_lib.mixers(), _lib.MIXERS_PROTOTYPES)):
        assert [n for n in names if not hasattr(getattr(d, n), "otherwise")] == [n for n in names if n in (
            "nv_strerror", "nv_last_error", "nv_abi_version", "nv_set_tuning", "nv_get_tuning")]


@pytest.mark.parametrize("name,args", [("nv_attn_decode_workspace_bytes_chunked", (3, 16, 8, 128, 4096, 0)), ("nv_attn_decode_suggest_chunk", (64, 16, 8, 9000, 70000)),
                                       ("nv_attn_prefill_workspace_bytes", (1, 512, 512, 8192, 32, 8, 128)), ("nv_attn_decode_static_scratch_bytes", ())])
def test_results(dll, name, args):
    fn = getattr(dll, name)
    assert fn(*args) == fn.otherwise(*args)


def test_conversions_and_errors(dll):
    fn = dll.nv_attn_prefill_query_tiles
    args = (4, 8192, 2048, 2048, 16, 8)
    want = fn.otherwise(*args)
    assert want > 0 and fn(*args) == want
    assert fn(4, 8192, 2048, 2048, 16, C.c_int(8)) == want                  # a ctypes object
    assert fn(4, 8192, 2048, (1 << 32) + 2048, 16, 8) == want               # what ctypes cuts to 32 bits
    assert fn(True, 8192, 2048, 2048, 16, 8) == fn.otherwise(True, 8192, 2048, 2048, 16, 8)
    for bad in ((4, 8192, 2048, 2048, 16), (4, 8192, 2048, 2048, 16, "8"), (4, 8192, 2048, 2048, 16, 8.0)):
        errors = []
        for f in (fn, fn.otherwise):
            with pytest.raises((TypeError, C.ArgumentError)) as e:
                f(*bad)
            errors.append(type(e.value))
        assert errors[0] is errors[1]


def test_pointers_floats_and_error_codes(dll):
    """A call that the host refuses before anything is launched: null pointers, 64-bit addresses, a float, a message."""
    fn = dll.nv_rmsnorm
    assert fn(None, None, None, 4, 128, 128, 1e-6, None) == fn.otherwise(None, None, None, 4, 128, 128, 1e-6, None) != 0
    assert fn(1 << 63, (1 << 64) - 16, None, 4, 128, 128, 1e-6, 0) != 0
    with pytest.raises(_lib.NanoVllmHipError):
        _lib.check(fn(None, None, None, 4, 128, 128, 1e-6, None), "nv_rmsnorm")
    assert fn(None, None, None, 0, 128, 128, 1, None) == fn.otherwise(None, None, None, 0, 128, 128, 1, None)      # an integer for a float


def test_only_callables_of_the_same_signature(dll, monkeypatch):
    """A module that was built from another header, or before modules said what they were built from, takes no call."""
    module = _lib._native_calls()
    name = "nv_attn_decode_suggest_chunk"

    class Other:
        bind = staticmethod(module.bind)

        @staticmethod
        def signature(n):
            s = module.signature(n)
            return s[:-1] + "i" if n == name else s           # its last argument was 32 bits then

    class Before:
        bind = staticmethod(module.bind)

    quick = lambda d, n: hasattr(getattr(d, n), "otherwise")
    monkeypatch.setattr(_lib, "_native_calls", lambda: Other)
    d = _lib.load()
    assert not quick(d, name) and quick(d, "nv_rmsnorm")
    monkeypatch.setattr(_lib, "_native_calls", lambda: Before)
    assert not any(quick(_lib.load(), n) for n in _lib.PROTOTYPES)
    monkeypatch.undo()
    turned = dict(_lib.PROTOTYPES, nv_rmsnorm=(C.c_int, [C.c_void_p] * 4 + [C.c_int64] * 3 + [C.c_float]))
    assert not quick(_lib.load(None, turned), "nv_rmsnorm")     # prototypes of the caller's own
    assert module.signature("nv_rmsnorm") == "ippplilfp" and module.signature("nv_strerror") is None
