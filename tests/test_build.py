"""The library's Makefile rebuilds what a change of a source, of a header or of
the rules makes stale (make -n in an object directory of its own)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "rapt_amd", "csrc")
OBJECTS = ["rapt_tracer", "rapt_tracer_f32", "rapt_bounce", "rapt_gcn", "rapt_mlp",
           "rapt_mlp_infer", "rapt_diag", "rapt_copy", "rapt_jit"]


@pytest.fixture
def built(tmp_path):
    """A copy of the sources and an object directory that is up to date."""
    shutil.copytree(CSRC, tmp_path / "rapt_amd" / "csrc")
    shutil.copytree(os.path.join(ROOT, "include"), tmp_path / "include")
    obj = tmp_path / "rapt_amd" / "lib" / "obj"
    obj.mkdir(parents=True)
    for path in [p for p in tmp_path.rglob("*") if p.is_file()]:
        os.utime(path, (1e9, 1e9))
    for k, name in enumerate(["rapt_jit_headers.inc"] + [o + s for s in (".o", ".d")
                                                         for o in OBJECTS]):
        dep = "rapt_gcn_kernel.hpp" if name == "rapt_gcn.d" else ""
        (obj / name).write_text("%s: %s\n" % ("../lib/obj/rapt_gcn.o", dep) if dep else "")
        os.utime(obj / name, (1e9 + 10 + k, 1e9 + 10 + k))
    lib = obj.parent / "librapt_hip.so"
    lib.write_text("")
    os.utime(lib, (1e9 + 100, 1e9 + 100))
    return tmp_path


def _compiled(tree):
    out = subprocess.run(["make", "-n", "-C", str(tree / "rapt_amd" / "csrc")],
                         capture_output=True, text=True, check=True).stdout
    return sorted(o for o in OBJECTS if "/%s.o %s.hip" % (o, o) in out)


def test_nothing_to_do(built):
    assert _compiled(built) == []


def test_object_without_a_list_of_its_headers(built):
    for o in ("rapt_gcn", "rapt_jit"):
        (built / "rapt_amd" / "lib" / "obj" / (o + ".d")).unlink()
    assert _compiled(built) == ["rapt_gcn", "rapt_jit"]


def test_changed_header_and_rules(built):
    csrc = built / "rapt_amd" / "csrc"
    os.utime(csrc / "rapt_gcn_kernel.hpp", (1e9 + 200, 1e9 + 200))
    assert "rapt_gcn" in _compiled(built)
    os.utime(csrc / "Makefile", (1e9 + 200, 1e9 + 200))
    assert _compiled(built) == sorted(OBJECTS)
