"""Runs library calls without a device: the HIP runtime replaced by
hip_host_stub.cpp (launches do nothing and are written down, allocations can be
made to fail).  A check runs in a process of its own:

    python -m tests._hoststub STUB.so MODULE FUNCTION
"""
import ctypes
import importlib
import os
import subprocess
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


class Stub:
    def __init__(self, path):
        self.lib = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)   # before the library that uses it
        self.lib.stub_launches.restype = ctypes.c_char_p
        self.lib.stub_fail_at.argtypes = [ctypes.c_long]
        for f in (self.lib.stub_allocations, self.lib.stub_held, self.lib.stub_peak):
            f.restype = ctypes.c_size_t

    def launches(self, call):
        """What `call` launches, a line each."""
        self.lib.stub_clear()
        call()
        return self.lib.stub_launches().decode().splitlines()

    def fails(self, call, k):
        """Whether `call` reports an error when its k-th allocation fails."""
        from helios_amd import capi
        self.lib.stub_fail_at(k)
        try:
            call()
            return False
        except capi.HccError:
            return True
        finally:
            self.lib.stub_fail_at(0)

    def each_failure(self, make, call, then=None):
        """`call` on what `make` gives, once for each of its allocations with that
        one failing: it reports an error, and afterwards `then` (the same call
        again, by default) launches what it does where nothing failed."""
        then = then or call
        obj = make()
        first = self.lib.stub_allocations()
        call(obj)
        count = self.lib.stub_allocations() - first
        assert count > 0, "no allocation in the call"
        fresh = obj if then is call else make()
        want = self.launches(lambda: then(fresh))
        for k in range(1, count + 1):
            obj = make()
            assert self.fails(lambda: call(obj), k), f"allocation {k} of {count}: failure not reported"
            got = self.launches(lambda: then(obj))
            assert got == want, f"allocation {k} of {count} failed, then {len(got)} launches: " + \
                "; ".join(f"{g} (expected {w})" for g, w in zip(got, want) if g != w)[:600]
        return count


def molecule(n, o):
    return dict(C=np.eye(n), F=np.eye(n), G=np.eye(n), nocc=o, eref=0.0)


def build(folder):
    lib = os.path.join(str(folder), "hip_host_stub.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-o", lib,
                    os.path.join(ROOT, "tests", "hip_host_stub.cpp")], check=True)
    return lib


def check(lib, function):
    """Runs FUNCTION(stub) of its module in a fresh process; fails with its output."""
    r = subprocess.run([sys.executable, "-m", "tests._hoststub", lib,
                        "tests." + function.__module__.split(".")[-1], function.__name__], cwd=ROOT,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, f"exit status {r.returncode}\n{r.stdout[-3000:]}"


if __name__ == "__main__":
    stub = Stub(sys.argv[1])
    getattr(importlib.import_module(sys.argv[2]), sys.argv[3])(stub)
