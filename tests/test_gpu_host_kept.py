"""Kept tables behind the C++ classes: what a program does between two searches or two top-Ks."""
import pytest

from test_host_gpu import run_exe

pytestmark = pytest.mark.gpu


def test_knn_matrices_that_a_program_works_on_itself():
    rc, out = run_exe("test_knn_gpu")
    assert rc == 0 and "0 failed" in out, out[-3000:]
