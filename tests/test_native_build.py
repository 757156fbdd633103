"""The native files are put in place whole, and an extension built for something else is refused."""

import os
import shutil
import subprocess
import sys

import pytest

from odc_amd import _native


def test_a_build_replaces_its_target_in_one_step(tmp_path):
    target = tmp_path / "lib.so"
    target.write_text("old")
    write = "import sys; open(sys.argv[1], 'w').write('half'); sys.exit(int(sys.argv[2]))"
    for status, text in ((3, "old"), (0, "half")):  # a failed build leaves what was there
        def command(output):
            assert output.parent == tmp_path and output != target  # same file system, another name
            return [sys.executable, "-c", write, str(output), str(status)]

        if status:
            with pytest.raises(RuntimeError, match="exit code 3"):
                _native._compile(target, command, False)
        else:
            assert _native._compile(target, command, False) == target
        assert target.read_text() == text and os.listdir(tmp_path) == ["lib.so"]


def test_every_builder_goes_through_it(monkeypatch):
    made = []
    monkeypatch.setattr(_native, "_compile", lambda target, command, verbose: made.append((target, command(target))) or target)
    for build in (_native.build_library, _native.build_ceiling_library, _native.build_torch_binding):
        build()
    assert [t.name for t, _ in made] == ["libodc_hip.so", "libodc_ceiling.so", "odc_torch.so"]
    for target, command in made:
        assert command[command.index("-o") + 1] == str(target)


def _load_in_a_child(path, patch=""):
    code = f"from odc_amd import _native; from pathlib import Path; {patch}; _native._load_torch_binding_file(Path({str(path)!r}))"
    return subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=_native.CSRC_DIR.parent.parent)


@pytest.mark.parametrize("patch,what", [
    ("_native.ABI_VERSION += 1", "ABI"),
    ("import torch; torch.__version__ = '0.0.1'", "torch 0.0.1"),
    ("import sys; sys.version_info = type('v', (), {'major': 3, 'minor': 99})", "CPython 3.99"),
])
def test_an_extension_built_for_something_else_is_refused(patch, what):
    _native.load_torch_binding()  # built when missing
    assert _load_in_a_child(_native.TORCH_BINDING_PATH, "pass").returncode == 0
    proc = _load_in_a_child(_native.TORCH_BINDING_PATH, patch)
    assert proc.returncode != 0 and "is stale" in proc.stderr and what in proc.stderr, proc.stderr


def test_a_file_that_is_no_library_is_an_import_error(tmp_path):
    path = tmp_path / "odc_torch.so"
    shutil.copy(_native.TORCH_BINDING_SOURCE, path)
    proc = _load_in_a_child(path, "pass")
    assert "ImportError" in proc.stderr and "cannot be loaded" in proc.stderr, proc.stderr
