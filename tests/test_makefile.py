"""The library's Makefile records the headers of every object, with any flags,
and compiles objects of an older Makefile again."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "2_amd", "csrc")


def _make(build, *args):
    r = subprocess.run(["make", "-n", "-C", CSRC, "BUILD=%s/" % build, "OUT=%s/lib.so" % build, *args],
                       capture_output=True, text=True, check=True)
    return [line for line in r.stdout.splitlines() if " -c " in line]


def test_every_object_records_its_headers(tmp_path):
    lines = _make(tmp_path, "CXXFLAGS=-O0")
    sources = [f for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp"))]
    assert len(lines) == len(sources)
    assert all("-MMD" in line for line in lines)


def test_objects_without_headers_are_compiled_again(tmp_path):
    names = [line.split(" -o ")[1].strip() for line in _make(tmp_path)]
    for o in names:
        open(o, "w").close()
        os.utime(o, (1, 1))
    # newer than every source, older than the Makefile
    newest = max(os.path.getmtime(os.path.join(CSRC, f)) for f in os.listdir(CSRC) if f != "Makefile")
    for o in names:
        os.utime(o, (newest + 1, newest + 1))
    assert len(_make(tmp_path, "-W", os.path.join(CSRC, "Makefile"))) == len(names)
    assert _make(tmp_path, "-o", os.path.join(CSRC, "Makefile")) == []
