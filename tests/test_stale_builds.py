"""Built files of other sources raise RuntimeError when they are loaded."""

from __future__ import annotations

import subprocess
import sysconfig

import pytest
import torch

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


MODULE = """
#include <Python.h>
static struct PyModuleDef def = {PyModuleDef_HEAD_INIT, "_pcpa_fast_calls", NULL, -1, NULL};
PyMODINIT_FUNC PyInit__pcpa_fast_calls(void) {
    PyObject* m = PyModule_Create(&def);
    %s
    return m;
}
"""


@pytest.mark.parametrize("source,message", [
    (MODULE % "", "rebuild"),
    (MODULE % 'PyModule_AddIntConstant(m, "version", %d); PyModule_AddStringConstant(m, "torch_version", "1.0");'
     % _native.FAST_CALLS_VERSION, "torch 1.0.*rebuild"),
    (MODULE % 'PyModule_AddIntConstant(m, "version", 0); PyModule_AddStringConstant(m, "torch_version", "%s");'
     % torch.__version__, "version 0.*rebuild"),
    # against torch libraries that are not these ones
    ("void absent_symbol(void);" + MODULE % "absent_symbol();", "rebuild"),
])
def test_extension_of_other_sources(source, message, tmp_path, monkeypatch):
    _compiled(tmp_path, source, "_pcpa_fast_calls.so", args=["-I" + sysconfig.get_paths()["include"]])
    monkeypatch.setattr(_native, "_fast_calls", None)
    monkeypatch.setattr(_native, "LIB_DIR", tmp_path)
    with pytest.raises(RuntimeError, match=message):
        _native.fast_calls()
    assert _native._fast_calls is None


def test_present_extension_loads():
    module = _native.fast_calls()
    assert (module.version, module.torch_version) == (_native.FAST_CALLS_VERSION, torch.__version__)
