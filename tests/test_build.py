"""CPU checks of the build script: what it links, and in which order, when a part is missing.
The compiler is stood in for by a function that records its output files."""
from __future__ import annotations

import importlib.util
import subprocess
from pathlib import Path

import pytest

PKG = Path(__file__).resolve().parent.parent / "mbr-cuda-tile_amd"


@pytest.fixture
def pkg_build(monkeypatch):
    spec = importlib.util.spec_from_file_location("mbrt_build_under_test", PKG / "build.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)

    def run(cmd, verbose):
        if any(c.endswith(mod.fail) for c in cmd if mod.fail):
            raise RuntimeError("command failed")
        Path(cmd[cmd.index("-o") + 1]).touch()

    mod.fail = ""
    monkeypatch.setattr(mod, "_run", run)
    return mod


def test_build_links_everything(pkg_build, tmp_path):
    out = pkg_build.build(out_dir=tmp_path)
    assert set(out) == {"libmbrt", "libmbrt_tensor", "mbrt_calls"} and all(p.exists() for p in out.values())
    torch = pytest.importorskip("torch")
    from mbrt import _abi

    assert out["mbrt_calls"].name == _abi.calls_path(torch.__version__).name  # the name that is loaded


def test_build_without_torch_links_the_libraries(pkg_build, tmp_path, monkeypatch, capsys):
    find = importlib.util.find_spec
    monkeypatch.setattr(importlib.util, "find_spec", lambda n, *a: None if n == "torch" else find(n, *a))
    out = pkg_build.build(out_dir=tmp_path)
    assert set(out) == {"libmbrt", "libmbrt_tensor"} and all(p.exists() for p in out.values())
    assert "native calls are not built: torch not found" in capsys.readouterr().out


def test_build_without_python_headers_links_the_libraries(pkg_build, tmp_path, monkeypatch, capsys):
    monkeypatch.setattr(pkg_build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert set(pkg_build.build(out_dir=tmp_path)) == {"libmbrt", "libmbrt_tensor"}
    assert "Python's headers not found" in capsys.readouterr().out


def test_build_error_in_the_extension_comes_after_the_libraries(pkg_build, tmp_path):
    pkg_build.fail = "calls.cpp"
    with pytest.raises(RuntimeError, match="command failed"):
        pkg_build.build(out_dir=tmp_path)
    assert (tmp_path / "libmbrt.so").exists() and (tmp_path / "libmbrt_tensor.so").exists()


@pytest.mark.parametrize("cpb,ok", [(0, False), (17, False), (1, True)])
def test_chunk_channels_per_block_out_of_range_do_not_build(pkg_build, cpb, ok):
    """A block of no waves, or of more than 1024 threads, is refused when it is compiled."""
    cmd = [pkg_build.HIPCC, *pkg_build.COMMON, f"-DMBRT_CHUNK_CPB={cpb}", "-x", "hip", "--cuda-host-only",
           "-fsyntax-only", str(PKG / "csrc" / "k_chunk.hip")]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert (r.returncode == 0) == ok, r.stderr
    assert ok or "one wave per channel" in r.stderr
