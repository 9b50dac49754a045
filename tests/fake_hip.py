"""The host side of the device library without a GPU: runs a function of a test
in a process of its own in which the library's HIP calls go to fake_hip.cc,
which keeps "device" memory on the host and notes kernel launches instead of
running them.  The caller asserts on what the function returns (JSON)."""
import ctypes
import functools
import inspect
import json
import os
import subprocess
import sys
import tempfile
import textwrap
from pathlib import Path

HERE = Path(__file__).resolve().parent
ROOT = HERE.parent
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@functools.cache
def _library():
    tmp = tempfile.TemporaryDirectory()
    so = Path(tmp.name) / "libfake_hip.so"
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-shared",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'lulesh_amd' / 'csrc'}", str(HERE / "fake_hip.cc"),
                    "-o", str(so)], check=True)
    return tmp, so  # removed with the test process


def run(function, *args):
    """function(fake, la, *args) in a process with the fake runtime; its source
    stands on its own (it may use what fake and la offer and import the rest)."""
    body = textwrap.dedent(inspect.getsource(function))
    script = (f"import sys; sys.path[:0] = [{str(HERE)!r}, {str(ROOT)!r}]\n"
              f"import json, fake_hip\nfake = fake_hip.Fake({str(_library()[1])!r})\n"
              f"import lulesh_amd as la\n{body}\n"
              f"print('RESULT ' + json.dumps({function.__name__}(fake, la, *json.loads({json.dumps(args)!r}))))\n")
    out = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout[-2000:] + out.stderr[-4000:]
    return json.loads(next(l for l in out.stdout.splitlines() if l.startswith("RESULT "))[7:])


class Fake:
    def __init__(self, so):
        # into the global scope, which the library's own dependencies come after
        self.lib = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
        self.lib.fake_launches.restype = ctypes.c_char_p
        self.lib.fake_fail_malloc_after.argtypes = [ctypes.c_long]
        self.lib.fake_copies.restype = ctypes.c_long

    def launches(self, grids=False):
        """Names of the kernels launched since the last call, without the
        namespace, e.g. k_nodal_brick<PolicyFp64, 256, false>; with their
        grid and block sizes."""
        lines = [l.removeprefix("void ") for l in self.lib.fake_launches().decode().replace("lgpu::", "").splitlines()]
        return lines if grids else [l.rsplit(" ", 2)[0] for l in lines]

    def fail_malloc_after(self, n):
        self.lib.fake_fail_malloc_after(n)

    def eos_slots(self):
        """(pos, count, rep, share) of the last k_eos launch's workgroups."""
        p = ctypes.POINTER(ctypes.c_int32)()
        n = self.lib.fake_eos_slots(ctypes.byref(p))
        return [tuple(p[4 * i:4 * i + 4]) for i in range(n)]

    def pinned(self, nbytes):
        p = ctypes.c_void_p()
        assert self.lib.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(nbytes), 0) == 0
        return p

    def copies(self):
        return self.lib.fake_copies()
