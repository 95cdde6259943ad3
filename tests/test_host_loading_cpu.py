"""The native host path where it cannot be used: its extension is missing, does not load or belongs to another torch.  Calls take the
general path then, with its results and its errors; host tensors, which both refuse, show which one answered.  And the C libraries
build where no Python with torch is found."""
import os
import subprocess

import pytest
import torch

from fusedswiglu_amd import FusedSwiGLU, _abi, _host, ops

CSRC = os.path.dirname(_abi.LIBRARY_PATH)


@pytest.fixture
def fresh(monkeypatch):
    monkeypatch.setattr(_host, "_module", None)
    return monkeypatch


def calls():
    x, w = torch.zeros(2, 8, dtype=torch.bfloat16), torch.zeros(8, 8, dtype=torch.bfloat16)
    return (lambda: FusedSwiGLU.apply(x, w, w), lambda: ops.swiglu(x, w, w), lambda: ops.swiglu_packed(x, w), lambda: ops.down_proj(x, w))


def missing(m, tmp_path):
    m.setattr(_host, "PATH", str(tmp_path / "_fsw_host.so"))


def broken(m, tmp_path):
    path = tmp_path / "_fsw_host.so"
    path.write_bytes(b"no shared object")
    m.setattr(_host, "PATH", str(path))


def other_torch(m, tmp_path):
    m.setattr(torch, "__version__", "1.0.0+rocm")


@pytest.mark.parametrize("how", [missing, broken, other_torch])
def test_calls_take_the_general_path(fresh, tmp_path, how):
    how(fresh, tmp_path)
    for i, call in enumerate(calls()):
        if i == 0:
            with pytest.warns(RuntimeWarning, match="cannot be used"), pytest.raises(AssertionError, match="HIP GPU"):
                call()
        with pytest.raises(AssertionError, match="HIP GPU"):
            call()
    x = torch.zeros(2, 8, dtype=torch.bfloat16)
    assert _host.swiglu(x, x, x) is None and _host.down_proj(x, x, False) is None


def test_before_the_library_is_built(fresh, tmp_path):
    """Errors of the arguments come first, as on the general path; nothing is remembered."""
    fresh.setattr(_abi, "_lib", None)
    fresh.setattr(_abi, "LIBRARY_PATH", str(tmp_path / "libfusedswiglu.so"))
    for call in calls():
        with pytest.raises(AssertionError, match="HIP GPU"):
            call()
    fresh.undo()
    assert _host.load().__name__ == "_fsw_host"


def test_the_extension_that_is_built_is_used():
    assert _host.load().__name__ == "_fsw_host" and _host.load().torch_version == torch.__version__.split("+")[0]


@pytest.mark.parametrize("python,built", [("/bin/false", False), ("/nonexistent/python3", False), ("python3", True)])
def test_make_without_torch(python, built):
    r = subprocess.run(["make", "-C", CSRC, "-n", "-B", f"PYTHON={python}"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    lines = r.stdout.splitlines()
    assert any("-o libfusedswiglu.so" in l for l in lines) and any("-o _fsw_host.so" in l for l in lines) == built
