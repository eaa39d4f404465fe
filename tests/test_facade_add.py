"""mrcpp::add of a FunctionTreeVector whose output is one of its terms (tests/cxx/add_into_term.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.gpu
def test_output_among_the_terms(tmp_path):
    from mrchem_amd import _lib
    exe, libdir = tmp_path / "add_into_term", os.path.dirname(_lib.LIB_PATH)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "cxx", "add_into_term.cpp"), "-L", libdir, "-lmwgreen",
                    "-Wl,-rpath," + libdir, "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "add into a term: ok" in r.stdout
