"""Build: a file's compiler-internal options are left out where the compiler does not know them; other errors stay errors."""
import pytest

from trida_stack_amd import build as B


def test_unknown_internal_option(tmp_path, monkeypatch, capsys):
    src = tmp_path / "unit.hip"
    src.write_text("int unit() { return 0; }\n")
    monkeypatch.setattr(B, "OBJ", tmp_path)
    monkeypatch.setattr(B, "FILE_FLAGS", {"unit": ["-mllvm", "-amdgpu-no-such-option=1"]})
    assert B._compile(src).stat().st_size > 0
    assert "-amdgpu-no-such-option" in capsys.readouterr().out
    src.write_text("int unit() { return }\n")
    with pytest.raises(RuntimeError, match="hipcc failed"):
        B._compile(src)
