"""What build() compiles first, and what is left where a part of it cannot be built."""
import pytest

from quantfour_adamw_cuda_amd import build as q4build


def test_the_host_module_stops_no_library(monkeypatch, tmp_path):
    """The C libraries need neither g++ nor torch's headers; where these are missing, build() says so after both are there, and
    a module of older sources is not left beside them."""
    built = []
    stale = tmp_path / "_q4host.so"
    stale.write_bytes(b"older sources")
    monkeypatch.setattr(q4build, "HOST_MODULE", str(stale))
    monkeypatch.setenv("CXX", str(tmp_path / "no such compiler"))
    monkeypatch.setattr(q4build, "compile_library", lambda out, sources, **kw: built.append(out))
    with pytest.raises((RuntimeError, OSError)):
        q4build.build()
    assert built == [q4build.LIB, q4build.PROBE_LIB]
    assert not stale.exists()
