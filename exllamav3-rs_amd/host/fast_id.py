"""What exl3r/_fast.so is built against, one line each: torch's folder and the Python headers' folder.  Fails where
either is missing.  torch is found without importing it."""
import importlib.util
import os
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
print(torch, include, sep="\n")
