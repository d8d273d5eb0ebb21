"""Built files of other sources raise RuntimeError when they are loaded."""

from __future__ import annotations

import subprocess

import pytest

from aws_training_study_amd import _native


def _compiled(tmp_path, source: str, name: str, compiler: str = "gcc", args=()):
    path = tmp_path / (name + ".c")
    path.write_text(source)
    subprocess.run([compiler, "-shared", "-fPIC", *args, str(path), "-o", str(tmp_path / name)], check=True)
    return tmp_path / name


@pytest.mark.parametrize("source,message", [
    # the present version, before some of its entries were added
    ("int pcpa_abi_version(void) { return %d; } void pcpa_absmax_bf16(void) {}" % _native.ABI_VERSION,
     "lacks .*pcpa_absmax_pair_bf16.*rebuild"),
    ("int pcpa_abi_version(void) { return %d; }" % (_native.ABI_VERSION - 1), "ABI version .*rebuild"),
    ("int unrelated;", "rebuild"),
])
def test_library_of_other_sources(source, message, tmp_path, monkeypatch):
    path = _compiled(tmp_path, source, "libstale.so")
    monkeypatch.setattr(_native, "_lib", None)
    monkeypatch.setattr(_native, "library_path", lambda: path)
    with pytest.raises(RuntimeError, match=message):
        _native.load_library()
    assert _native._lib is None
