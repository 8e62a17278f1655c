"""The native host side of calls: loaded with the library, and everything but plain device tensors is left to Python."""
import os
import shutil
import subprocess
import sysconfig
import warnings

import pytest
import torch


def test_native_calls_leave_the_rest_to_python():
    from vllm_hymeta import _C
    _C.load()
    if _C.calls is None:
        pytest.skip("hymeta_calls.so is not built")
    q, starts = torch.zeros(2, 4, 128, dtype=torch.bfloat16), torch.zeros(3, dtype=torch.int32)
    state, decay = torch.zeros(2, 4, 128, 128), torch.ones(4)
    for args in ((), (q,), (None,) * 13, (q, q, q, state, starts, starts, starts, 1, decay, None, None, None, 0), ("q", 1, 2.0),
                 (q.numpy,) * 13, (torch.nn.Parameter(q.float()),) * 13):
        assert _C.calls.decay_scan(*args) is None
    for name in ("sink_attention", "meta_swa_paged_decode", "meta_swa_prefill", "lightning_attention", "delta_rule"):
        assert getattr(_C.calls, name)(*[q] * 26) is None and getattr(_C.calls, name)() is None
    with pytest.raises(TypeError):
        _C.calls.setup(_C)


UNRESOLVED = "extern void not_in_this_torch(void); void *PyInit_hymeta_calls(void) { not_in_this_torch(); return 0; }"
OLDER = """
#include <Python.h>
static struct PyModuleDef def = {PyModuleDef_HEAD_INIT, "hymeta_calls", 0, -1, 0};
PyMODINIT_FUNC PyInit_hymeta_calls(void) {
  PyObject *m = PyModule_Create(&def);
  PyModule_AddObject(m, "built_for", Py_BuildValue("(ssi)", "2.0.0 another", "3.10", 9));
  return m;
}
"""


@pytest.mark.parametrize("source,says", [(UNRESOLVED, "does not load"), (OLDER, "is built for")], ids=["unresolved", "older"])
def test_native_calls_of_another_torch_count_as_absent(tmp_path, monkeypatch, source, says):
    from vllm_hymeta import _C
    (tmp_path / "calls.c").write_text(source)
    if shutil.which("gcc") is None or not os.path.exists(os.path.join(sysconfig.get_paths()["include"], "Python.h")):
        pytest.skip("no gcc or no Python.h")
    subprocess.run(["gcc", "-shared", "-fPIC", "-Wl,-z,now", "-I", sysconfig.get_paths()["include"], str(tmp_path / "calls.c"), "-o", str(tmp_path / "hymeta_calls.so")], check=True)
    monkeypatch.setattr(_C, "_CALLS_NAME", str(tmp_path / "hymeta_calls.so"))      # (an absolute path stands for itself)
    monkeypatch.setattr(_C, "_lib", None)
    monkeypatch.setattr(_C, "calls", None)
    with pytest.warns(RuntimeWarning, match=says):
        lib = _C.load()
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _C.load() is lib and _C.calls is None
    assert lib.hymeta_abi_version() == _C.ABI_VERSION


@pytest.mark.parametrize("lacks", ["CXX=no-such-compiler", "PYTHON=no-such-python"])
def test_the_library_is_made_without_what_the_calls_need(tmp_path, lacks):
    """The rule of the native calls alone, in a folder of its own (the library's objects are not made again)."""
    package = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-hymeta_amd")
    if shutil.which("make") is None:
        pytest.skip("no make")
    made = tmp_path / "hymeta_calls.so"
    made.write_text("of an earlier torch")
    os.utime(made, (1, 1))
    run = subprocess.run(["make", "-C", package, lacks, f"OBJDIR={tmp_path}", f"CALLS={made}", str(made)], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and "the package works without it" in run.stderr and not made.exists()
