"""libqgemm.so does not depend on _fast.so: it is built and used without it."""
import importlib

import pytest
import torch


def test_library_is_linked_without_the_native_calls(monkeypatch, tmp_path):
    """No csrc/host/fast.cpp to compile, and a _fast.so of an older build."""
    build = importlib.import_module("355_1_trans_amd.build")
    (tmp_path / "one.hip").write_text('extern "C" int one() { return 1; }\n')
    for name, path in (("CSRC", tmp_path), ("OUT_DIR", tmp_path / "_build"), ("LIB", tmp_path / "libqgemm.so"),
                       ("FAST", tmp_path / "_fast.so")):
        monkeypatch.setattr(build, name, path)
    build.FAST.write_bytes(b"old")
    with pytest.warns(UserWarning, match="_fast.so was not built"):
        assert build.build() == build.LIB
    assert build.LIB.exists() and not build.FAST.exists()


def test_native_calls_that_do_not_load_leave_the_wrappers(qgemm, monkeypatch, tmp_path):
    """A _fast.so that cannot be imported warns once; the Python code serves
    the calls.  While the library is missing nothing is settled."""
    monkeypatch.setattr(qgemm, "_PKG", tmp_path)
    monkeypatch.setattr(qgemm, "_fast", None)
    (tmp_path / "_fast.so").write_bytes(b"not a library")
    a = torch.zeros(16, 128, dtype=torch.uint8)
    with monkeypatch.context() as p:
        p.setattr(qgemm, "LIB_PATH", tmp_path / "libqgemm.so")
        assert qgemm.fast() is qgemm._NoFast and qgemm._fast is None
    with pytest.warns(UserWarning, match="_fast.so cannot be used"), pytest.raises(ValueError, match="GPU"):
        qgemm.gemm_a8w8_mxfp8(a, a, a[:, :4], a[:, :4])
    assert qgemm.fast() is qgemm._NoFast and qgemm._fast is qgemm._NoFast
