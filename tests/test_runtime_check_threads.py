"""The one-runtime check beside imports: a thread that asks for the count of loaded objects over and over
does not stop a thread that imports extension modules (the dynamic linker's lock and the interpreter's
are never taken in opposite orders).  CPU only."""
import os
import subprocess
import sys

import pytest

from cnhip import abi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "cressim-neo_amd")

BODY = """
import importlib.machinery, importlib.util, os, shutil, sys, threading
sys.path.insert(0, {pkg!r})
import cnhip
cnhip.load_library()
from cnhip import abi
import _queue
stop = threading.Event()
calls = [0, 0]

def ask(k):
    while not stop.is_set():
        abi.objects_loaded()
        abi.require_single_hip_runtime('thread')
        calls[k] += 1

threads = [threading.Thread(target=ask, args=(k,), daemon=True) for k in range(2)]
for t in threads:
    t.start()
before = abi.objects_loaded()
for k in range(150):
    # a file of its own each time, so that the linker loads it
    path = os.path.join({tmp!r}, str(k), os.path.basename(_queue.__file__))
    os.makedirs(os.path.dirname(path))
    shutil.copy(_queue.__file__, path)
    loader = importlib.machinery.ExtensionFileLoader('_queue', path)
    spec = importlib.util.spec_from_file_location('_queue', path, loader=loader)
    importlib.util.module_from_spec(spec)
    print('import', k, flush=True)
after = abi.objects_loaded()
stop.set()
for t in threads:
    t.join()
print('LOADED', after - before, 'CALLS', min(calls) > 0)
"""


@pytest.mark.skipif(not os.path.exists(abi.LIB_PATH), reason="libcn_hip.so not built")
def test_imports_beside_the_runtime_check_do_not_hang(tmp_path):
    out = subprocess.run([sys.executable, "-c", BODY.format(pkg=PKG, tmp=str(tmp_path))], capture_output=True, text=True,
                         timeout=60, check=True).stdout
    assert "LOADED 150 CALLS True" in out
