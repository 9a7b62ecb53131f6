"""The extension's build."""
import os
import sys

sys.path.insert(0, os.path.join(os.path.dirname(__file__), ".."))
import build_ext


def test_a_changed_header_builds_every_kernel_again(tmp_path):
    """Its digest is a part of the compiler's command, and ninja runs a changed command."""
    (tmp_path / "args.h").write_text("struct Args { int a; };")
    (tmp_path / "kernel.hip").write_text("")
    first = build_ext.headers_digest(str(tmp_path))
    (tmp_path / "kernel.hip").write_text("// ninja sees this one by itself")
    assert build_ext.headers_digest(str(tmp_path)) == first
    (tmp_path / "args.h").write_text("struct Args { int more, a; };")
    assert build_ext.headers_digest(str(tmp_path)) != first
