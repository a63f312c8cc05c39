"""What exl3r/_fast.so is built for and against, one line each: its identity (torch's version and the interpreter's ABI
tag, as exl3r/_lib.py forms it), torch's folder and the Python headers' folder.  Fails where one of them is missing.
torch is found without importing it."""
import importlib.util
import os
import runpy
import sys
import sysconfig

spec = importlib.util.find_spec("torch")
if spec is None or not spec.origin:
    sys.exit("this interpreter has no torch")
torch = os.path.dirname(spec.origin)
include = sysconfig.get_paths()["include"]
for header in (os.path.join(torch, "include", "c10", "hip", "HIPStream.h"), os.path.join(include, "Python.h")):
    if not os.path.exists(header):
        sys.exit(f"{header} is missing")
version = runpy.run_path(os.path.join(torch, "version.py"))["__version__"]
print(f"{version} {sys.implementation.cache_tag}", torch, include, sep="\n")
