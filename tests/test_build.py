"""Which objects an incremental build compiles again (a stand-in for the compiler writes the flags it
was called with into the object)."""
import os

import pytest

from cedar_amd import build as B


@pytest.fixture
def tree(tmp_path, monkeypatch):
    src = tmp_path / "csrc"
    src.mkdir()
    (tmp_path / "include").mkdir()
    (tmp_path / "include" / "a.h").write_text("")
    (src / "b.hpp").write_text("")
    (src / "one.hip").write_text("")
    (src / "two.cpp").write_text("")
    cc = tmp_path / "cc"
    cc.write_text("#!/bin/sh\nwhile [ $# -gt 0 ]; do case $1 in -o) out=$2;; -D*) d=$1;; esac; shift; done\n"
                  "[ \"$d\" = -DFAIL ] && exit 1\necho built $d >> $out\n")
    cc.chmod(0o755)
    for k, v in dict(HERE=str(tmp_path / "pkg"), CSRC=str(src), OBJDIR=str(tmp_path / "obj"),
                     HIPCC=str(cc), FLAGS=["-DX"]).items():
        monkeypatch.setattr(B, k, v)
    os.mkdir(B.OBJDIR)
    for f in (tmp_path / "include" / "a.h", src / "b.hpp", src / "one.hip", src / "two.cpp"):
        os.utime(f, (1, 1))
    return src


def objects(incremental=True):
    """The flags of each compilation so far, per source."""
    return [open(B._compile(s, incremental)).read().split("\n")[:-1] for s in ("one.hip", "two.cpp")]


def test_incremental_build(tree):
    assert objects() == [["built -DX"]] * 2
    assert objects() == [["built -DX"]] * 2  # nothing changed
    os.utime(tree / "one.hip")
    os.utime(os.path.join(B.OBJDIR, "one.hip.o"), (2, 2))
    assert objects() == [["built -DX"] * 2, ["built -DX"]]
    assert objects(incremental=False) == [["built -DX"] * 3, ["built -DX"] * 2]


def test_changed_flags_compile_everything_again(tree, monkeypatch):
    objects()
    monkeypatch.setattr(B, "FLAGS", ["-DY"])
    assert objects() == [["built -DX", "built -DY"]] * 2
    assert objects() == [["built -DX", "built -DY"]] * 2


def test_failed_compilation_leaves_nothing_to_skip(tree, monkeypatch):
    objects()
    monkeypatch.setattr(B, "FLAGS", ["-DFAIL"])
    with pytest.raises(RuntimeError):
        objects()
    monkeypatch.setattr(B, "FLAGS", ["-DX"])
    assert objects()[0] == ["built -DX"] * 2


def test_objects_of_unknown_flags_are_compiled_again(tree):
    for s in ("one.hip", "two.cpp"):
        open(os.path.join(B.OBJDIR, s + ".o"), "w").write("built -DOLD\n")
    assert objects() == [["built -DOLD", "built -DX"]] * 2
