"""What the build takes for up to date (onnxruntime_amd/build.py).  Nothing is compiled here."""
import os

import pytest

from onnxruntime_amd import build as B


class Compiled(Exception):
    pass


@pytest.mark.parametrize("old,rebuilt", [((), False), (("LIB",), True), (("CALLS_LIB",), True), (("LIB", "CALLS_LIB"), True)])
def test_a_library_older_than_the_sources_is_built_again(monkeypatch, tmp_path, old, rebuilt):
    """A build whose last step, the native calls, failed leaves a new library beside old calls: both have to be new."""
    for name in ("LIB", "CALLS_LIB"):
        path = tmp_path / name
        path.write_bytes(b"")
        os.utime(path, (0, 0) if name in old else (2 ** 33, 2 ** 33))
        monkeypatch.setattr(B, name, path)

    def compile_one(*args):
        raise Compiled
    monkeypatch.setattr(B, "_compile", compile_one)
    if rebuilt:
        with pytest.raises(Compiled):
            B.build(force=False, jobs=1)
    else:
        assert B.build(force=False, jobs=1) == tmp_path / "LIB"
