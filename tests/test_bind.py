"""The Python calls into the library (csrc/bind.cpp): every declared entry
point, the C argument conversions, and errors reported on the same thread."""
import pytest

from serving import _native
from serving.fake_paged_attn import _bound


def test_every_entry_point_is_there():
    calls = _native.calls()
    for name in _native.EXPORTED:
        if name != "pkv_last_error":  # read through lib() by check()
            assert callable(getattr(calls, name)), name
    assert calls.pkv_version() == _native.lib().pkv_version()


def test_conversions():
    calls = _native.calls()
    args = (32, 1, 16, 1, 64, 64, 16, 0, 0, 2)
    assert (calls.pkv_attention_workspace_bytes(*args)
            == _native.lib().pkv_attention_workspace_bytes(*args) > 0)
    with pytest.raises(TypeError):
        calls.pkv_attention_workspace_bytes(*args[:-1])
    with pytest.raises(TypeError):
        calls.pkv_attention_workspace_bytes("32", *args[1:])
    with pytest.raises(OverflowError):
        calls.pkv_attention_workspace_bytes(1 << 40, *args[1:])


def test_null_pointers_and_last_error():
    rc = _native.calls().pkv_rms_norm(None, None, None, None, None, 1, 64, 64, 64, 1e-5, 2, None)
    assert rc == _native.PKV_ERR_INVALID
    with pytest.raises(ValueError, match="null"):
        _native.check(rc, "pkv_rms_norm")


def test_bounds_fit_the_librarys_int():
    """A context bound or partition length of any size is accepted (ctypes took
    its low 32 bits): past 2^30 tokens it bounds nothing."""
    args = lambda b: (32, 1, 16, 1, 64, 64, 16, b, 0, 2)  # noqa: E731
    size = _native.calls().pkv_attention_workspace_bytes
    for b in (1 << 31, (1 << 32) + 5, 1 << 40, 1 << 70):
        assert size(*args(_bound(b))) == size(*args(0))
    assert [_bound(b) for b in (-3, 0, 7, 1 << 30, 1 << 31)] == [-3, 0, 7, 1 << 30, 1 << 30]


@pytest.mark.parametrize("content", [None, b"not a shared object"])
def test_without_the_module_the_calls_go_through_ctypes(monkeypatch, tmp_path, content):
    path = tmp_path / "_pkvbind.so"
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(_native, "BIND_PATH", str(path))
    monkeypatch.setattr(_native, "_calls", None)
    assert _native.calls() is _native.lib()
    assert _native.calls().pkv_version() >= 1


def test_built_without_python_headers(monkeypatch, tmp_path, capsys):
    import build_native
    monkeypatch.setattr(build_native, "BIND", str(tmp_path / "_pkvbind.so"))
    monkeypatch.setattr(build_native, "CXX", "no-such-compiler")
    (tmp_path / "_pkvbind.so").write_bytes(b"stale")
    build_native.build_bind()
    assert "not built" in capsys.readouterr().out
    assert not (tmp_path / "_pkvbind.so").exists()
