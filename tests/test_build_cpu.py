"""The Makefile's optional target: exl3r/_fast.so, the native form of the Python wrappers, is built against the
interpreter's torch, and the library, whose hosts need no torch, is built without it where there is none."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "exllamav3-rs_amd")


@pytest.fixture
def tree(tmp_path):
    """The Makefile and the sources it reads, in a folder of their own."""
    pkg = tmp_path / "exllamav3-rs_amd"
    shutil.copytree(os.path.join(PKG, "host"), pkg / "host")
    shutil.copytree(os.path.join(PKG, "csrc"), pkg / "csrc")
    shutil.copytree(os.path.join(ROOT, "include"), tmp_path / "include")
    shutil.copy(os.path.join(PKG, "Makefile"), pkg)
    return pkg


def make(pkg, python, *targets):
    return subprocess.run(["make", "-C", str(pkg), f"PYTHON={python}", *targets], capture_output=True, text=True, timeout=600)


def no_torch(tmp_path, with_headers):
    """An interpreter that finds no torch, or one without HIP headers."""
    path = tmp_path / "site"
    if with_headers:
        (path / "torch").mkdir(parents=True)
        (path / "torch" / "__init__.py").write_text("")
        (path / "torch" / "version.py").write_text("__version__ = '2.0.0+cpu'\n")
    run = tmp_path / "python"
    run.write_text(f"#!/bin/sh\nPYTHONPATH={path} exec {sys.executable} -S \"$@\"\n")
    run.chmod(0o755)
    return run


@pytest.mark.parametrize("torch_of_cpu", [False, True])
def test_make_without_a_rocm_torch(tree, tmp_path, torch_of_cpu):
    r = make(tree, no_torch(tmp_path, torch_of_cpu), "exl3r/_fast.so")
    assert r.returncode == 0, r.stderr
    assert "skipped" in r.stdout
    assert not (tree / "exl3r" / "_fast.so").exists()


def test_module_follows_the_torch_it_is_built_for(tree, tmp_path):
    """Another torch version or interpreter tag builds the module again; the same ones do not."""
    (tree / "exl3r").mkdir()
    so, run = tree / "exl3r" / "_fast.so", no_torch(tmp_path, True)
    (tmp_path / "site" / "torch" / "include" / "c10" / "hip").mkdir(parents=True)
    (tmp_path / "site" / "torch" / "include" / "c10" / "hip" / "HIPStream.h").write_text("")
    compiler = tmp_path / "cxx"
    compiler.write_text("#!/bin/sh\necho \"$@\" >> %s\ntouch exl3r/_fast.so\n" % (tmp_path / "built"))
    compiler.chmod(0o755)
    built = lambda: (tmp_path / "built").read_text().splitlines()
    for version, builds in (("2.0.0", 1), ("2.0.0", 1), ("2.1.0", 2), ("2.1.0", 2)):
        (tmp_path / "site" / "torch" / "version.py").write_text(f"__version__ = {version!r}\n")
        r = make(tree, run, f"CXX={compiler}", "exl3r/_fast.so")
        assert r.returncode == 0 and so.exists(), r.stderr
        assert len(built()) == builds
        assert f'-DEXL3R_BUILT_FOR="{version} {sys.implementation.cache_tag}"' in built()[-1]
