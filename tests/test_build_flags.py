"""An object is compiled again when its source, a header or its flags change, and not otherwise (build.py)."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture
def build(monkeypatch):
    spec = importlib.util.spec_from_file_location("repo_build", os.path.join(ROOT, "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    mod.ran = []

    def run(cmd):
        mod.ran.append(cmd)
        open(cmd[-1], "w").write("object")
        return ""
    monkeypatch.setattr(mod, "_run", run)
    return mod


def test_other_flags_make_another_object(build, tmp_path, monkeypatch):
    src, header, obj = tmp_path / "k.hip", tmp_path / "h.h", tmp_path / "out" / "k.o"
    src.write_text("kernel")
    header.write_text("header")

    def compiled(extra=()):
        return build._compile_hip(src, obj, [header], False, extra)
    assert compiled() and not compiled()
    monkeypatch.setitem(build.FILE_FLAGS, "k", ["-mllvm", "-some-form"])
    assert compiled() and "-some-form" in build.ran[-1] and not compiled()
    monkeypatch.delitem(build.FILE_FLAGS, "k")
    assert compiled() and not compiled()
    assert compiled(["-DMORE"]) and not compiled(["-DMORE"])
    os.utime(header, (obj.stat().st_mtime + 5,) * 2)
    assert compiled(["-DMORE"])


def test_a_failed_compile_leaves_nothing_that_looks_up_to_date(build, tmp_path, monkeypatch):
    src, obj = tmp_path / "k.hip", tmp_path / "k.o"
    src.write_text("kernel")
    assert build._compile_hip(src, obj, [], False)

    def fail(cmd):
        raise SystemExit("build failed")
    good = build._run
    monkeypatch.setattr(build, "_run", fail)
    with pytest.raises(SystemExit):
        build._compile_hip(src, obj, [], False, ["-DOTHER"])
    monkeypatch.setattr(build, "_run", good)
    assert build._compile_hip(src, obj, [], False)
