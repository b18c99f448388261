"""The native circuit recorder is optional: the libraries build without Python's
headers, and circuits record the same without it (no GPU)."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "dgquest_amd")


def _targets(*args):
    out = subprocess.check_output(["make", "-n", "-B", "-C", PKG, *args], text=True)
    return {lib for lib in ("libdgq_engine.so", "libQuEST_f64.so", "libQuEST_f32.so", "libdgq_pyrecord.so") if f"-o {PKG}/lib/{lib}" in out}


def test_make_needs_no_python_headers(tmp_path):
    assert _targets() >= {"libdgq_engine.so", "libQuEST_f64.so", "libQuEST_f32.so"}
    assert _targets(f"PYINC={tmp_path}") == {"libdgq_engine.so", "libQuEST_f64.so", "libQuEST_f32.so"}


def test_circuits_record_the_same_without_it(tmp_path):
    for lib in ("libdgq_engine.so", "libQuEST_f64.so"):
        os.symlink(os.path.join(PKG, "lib", lib), tmp_path / lib)
    code = """
import sys
from dgquest_amd import circuits, quest as Q, serve as S
api = Q.QuEST(2, libdir=sys.argv[1])
r = S.record(api, 7, circuits.layered_u3_cz(7, 3, 1))
print(r.gates.tobytes().hex())
"""
    out = [subprocess.run([sys.executable, "-c", code, str(d)], capture_output=True, text=True, cwd=ROOT, timeout=120)
           for d in (tmp_path, os.path.join(PKG, "lib"))]
    for p in out:
        assert p.returncode == 0, p.stderr
    assert len(out[0].stdout) > 100 and out[0].stdout == out[1].stdout
