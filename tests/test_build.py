"""CPU: what counts as built.  ``csrc/build.py`` makes several files from several sources; each is compared with its own."""
import os

import pytest


@pytest.fixture
def built(tmp_path, monkeypatch):
    import sparse  # noqa: F401  (csrc on the path, everything built)
    import importlib.util
    from sparse.kernel import _CSRC
    spec = importlib.util.spec_from_file_location("csrc_build_under_test", os.path.join(_CSRC, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    paths = {name: str(tmp_path / name) for name in ("lib", "fences", "host")}
    for path in paths.values():
        open(path, "w").close()
    monkeypatch.setattr(build, "LIB", paths["lib"])
    monkeypatch.setattr(build, "CHECK_VARIANTS", {"fences": (paths["fences"], [])})
    monkeypatch.setattr(build, "HOST_CALLS", paths["host"])
    return build, paths


def test_each_file_is_compared_with_its_own_sources(built):
    build, paths = built
    assert not build.out_of_date()
    for path in paths.values():
        os.utime(path, (0, 0))                  # older than every source, the others new: a build that failed half way
        assert build.out_of_date()
        os.utime(path)
        assert not build.out_of_date()
        os.rename(path, path + ".away")
        assert build.out_of_date()
        os.rename(path + ".away", path)


def test_host_calls_of_another_library_or_torch_are_refused(monkeypatch):
    import ctypes

    import torch
    from sparse import _native, kernel
    other = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: 1)
    entries = {name: ctypes.cast(getattr(kernel.lib, name), ctypes.c_void_p).value for name in _native._ENTRIES}
    entries["bsa_version"] = ctypes.cast(other, ctypes.c_void_p).value
    with pytest.raises(ImportError, match="version"):
        kernel.host_calls.setup(entries, {}, {}, {})
    monkeypatch.setattr(torch, "__version__", "0.0")
    with pytest.raises(ImportError, match="torch"):
        kernel.load_host_calls()
