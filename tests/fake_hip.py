"""Runs of the host library on tests/fakehip/fake_hip.c, a HIP runtime without a
device: what is launched, how large, and what the library does when an
allocation is refused.  In a process of its own (`run`), because the runtime
calls of libamrgpu.so are bound when it is loaded."""
import ctypes as C
import os
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "fakehip", "fake_hip.c")
DEVICE, PINNED = 0, 1


def run(module, function, *args):
    """module.function(fake, *args) in a child process, with the fake runtime
    loaded; an exception there fails the caller."""
    with tempfile.TemporaryDirectory() as d:
        so = os.path.join(d, "libfakehip.so")
        subprocess.run(["gcc", "-O1", "-shared", "-fPIC", SRC, "-o", so], check=True)
        code = ("import sys, importlib; sys.path.insert(0, %r); from tests import fake_hip; "
                "fake = fake_hip.Fake(%r); getattr(importlib.import_module(%r), %r)(fake, *%r); "
                "print('child ok')" % (ROOT, so, module, function, args))
        r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT,
                           timeout=300)
    assert r.returncode == 0 and "child ok" in r.stdout, r.stdout + r.stderr


class Fake:
    def __init__(self, so):
        self.L = C.CDLL(so, mode=C.RTLD_GLOBAL)
        self.L.fake_name.restype = C.c_char_p
        self.L.fake_arg0.restype = C.c_uint64
        from amrclaw_amd import capi
        capi.lib()
        assert self.allocs(PINNED) == 0

    def clear(self):
        self.L.fake_clear()

    def launches(self, name=""):
        """(kernel name, workgroups along x, first argument) of the launches
        since clear() whose mangled name holds `name`."""
        out = [(self.L.fake_name(i).decode(), int(self.L.fake_grid(i)), int(self.L.fake_arg0(i)))
               for i in range(self.L.fake_launches())]
        return [x for x in out if name in x[0]]

    def refuse(self, kind, n):
        """Refuse the n-th allocation of the kind from now (0: none)."""
        self.L.fake_refuse(kind, n)

    def allocs(self, kind):
        return self.L.fake_allocs(kind)

    def live(self, kind):
        return self.L.fake_live(kind)
