"""The library's host code on the CPU, over a HIP runtime that runs nothing
(tests/fake_hip.c): which kernels a call launches, and with what arguments.
The fake must come first into a process, so a test runs its script in a
process of its own, with run(); the script calls load()."""
import ctypes as C
import glob
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HOOK = C.CFUNCTYPE(None, C.c_char_p, C.c_uint, C.POINTER(C.c_void_p))


def run(script: str, tmp_path, timeout: int = 100, lib: str = "") -> str:
    """`script` in a process whose HIP calls are the fake's; its output.
    lib: another library than the built one."""
    from neslgpu_amd import cvl
    if not os.path.exists(lib or cvl.LIB_PATH):
        pytest.skip("libcvl_hip.so not built (python -m neslgpu_amd.build)")
    if not shutil.which("gcc"):
        pytest.skip("no gcc")
    so = str(tmp_path / "libfakehip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "fake_hip.c")], check=True)
    r = subprocess.run([sys.executable, "-c", "import sys; from fake_hip import load, word, Post\n" + script],
                       env=dict(os.environ, FAKE_HIP=so, CVLHIP_LIBRARY=lib or cvl.LIB_PATH, PYTHONPATH=os.pathsep.join([HERE, os.path.dirname(HERE)])),
                       capture_output=True, text=True, timeout=timeout)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return r.stdout


def variant(tmp_path, source: str, key: str, value) -> str:
    """The library with one of the tuner's values for `source`, linked with
    the objects of the last build ("": it is the built one's)."""
    from neslgpu_amd import build as B, tune as T
    assert T.norm(value) in [T.norm(v) for v in T.SPACE[key][0]]
    if T.norm(value) == T.norm(T.key_value(key)):
        return ""
    objs = {os.path.basename(o): o for o in glob.glob(os.path.join(B.OBJ, "*.hip.o"))}
    if not os.path.exists(B.HIPCC) or source + ".o" not in objs:
        pytest.skip("no hipcc, or no objects of a build")
    objs[source + ".o"] = o = str(tmp_path / "variant.o")
    lib = str(tmp_path / "libcvl_hip.so")
    subprocess.run([B.HIPCC, *B.FLAGS, *B.extra_flags(), *T.defines(key, value), "-I", B.OBJ, "-c",
                    os.path.join(B.CSRC, source), "-o", o], check=True, capture_output=True)
    subprocess.run([B.HIPCC, f"--offload-arch={B.ARCH}", "-shared", "-fPIC", "-o", lib, *objs.values()], check=True)
    return lib


def load(on_launch):
    """(fake, library): on_launch(name, workgroups, args) is called for every
    kernel launch; args[i] is the address of argument i."""
    fake = C.CDLL(os.environ["FAKE_HIP"], mode=C.RTLD_GLOBAL)
    fake.fake_device_of.argtypes = [C.c_void_p]
    from neslgpu_amd.cvl import Lib
    lib = Lib()
    hook = HOOK(lambda name, wgs, args: on_launch(name.decode(), wgs, args))
    fake.fake_set_hook(hook)
    fake.keep = hook
    return fake, lib


def word(args, i, ty=C.c_uint64):
    """Argument i of a launch."""
    return C.cast(args[i], C.POINTER(ty))[0]


class Post(C.Structure):
    """The word a kernel posts to the host (cvl_hip.hpp, Mailbox)."""
    _fields_ = [("seq", C.c_uint64), ("value", C.c_uint64)]

    @staticmethod
    def to(mailbox: int, seq: int, value: int):
        p = Post.from_address(mailbox)
        p.value = value
        p.seq = seq
