"""The library's host runtime linked with a stand-in for HIP (tests/cxx/hip_stand_in.cpp): contexts on
a machine without a GPU, for tests of what the host does around the kernels.  Launches compute
nothing."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from spacetime_amd import gpe

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def build(out):
    cxx = shutil.which("g++")
    if cxx is None or not os.path.isdir("/opt/rocm/include/hip"):
        pytest.skip("needs g++ and the HIP headers")
    csrc = os.path.join(ROOT, "spacetime_amd", "csrc")
    subprocess.run([cxx, "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + csrc]
                   + [os.path.join(csrc, f) for f in ("gpe_host.cpp", "gpe_states.cpp", "gpe_io.cpp")]
                   + [os.path.join(ROOT, "tests", "cxx", "hip_stand_in.cpp"), "-Wl,-Bsymbolic", "-o", out], check=True)


class StandIn:
    """gpe.* on the stand-in library while active; what it counted."""

    def __init__(self, path):
        saved, gpe._LIB = gpe._LIB, None
        try:
            self.lib = gpe.load_library(path)
        finally:
            gpe._LIB = saved
        self.lib.stand_in_limits.argtypes = [ctypes.c_longlong, ctypes.c_longlong]

    def limits(self, capacity=1 << 40, max_block=1 << 40):
        self.lib.stand_in_limits(capacity, max_block)

    def counts(self):
        out = (ctypes.c_longlong * 5)()
        self.lib.stand_in_counts(out)
        return dict(zip(("allocs", "host_allocs", "copies", "used", "waves"), out))

    def reduction(self):
        out = (ctypes.c_longlong * 12)()
        self.lib.stand_in_reduction(out)
        return dict(zip(("nx", "ny", "nz", "V", "ty", "rows", "nseg", "waves", "ntile", "segs", "per", "blocks"), out))

    def sweep(self):
        out = (ctypes.c_longlong * 5)()
        self.lib.stand_in_sweep(out)
        return dict(zip(("rows", "x_per_lane", "tile_rows", "waves", "exchange"), out))


def started(lattice, ncomp, precision, dims, **kw):
    """A started context of a box."""
    cfg = gpe.Config.centred_box(lattice, dims, 0.7, ncomp=ncomp, precision=precision, dt=1e-4, **kw)
    st = gpe.Stepper(cfg)
    st.set_state(np.zeros(cfg.shape, dtype=np.complex128))
    st.start(gpe.START_EULER)
    return st


_PATH = None


@pytest.fixture
def stand_in(tmp_path_factory, monkeypatch):
    global _PATH
    if _PATH is None:
        _PATH = str(tmp_path_factory.mktemp("stand_in") / "libgpe_stand_in.so")
        build(_PATH)
    s = StandIn(_PATH)
    monkeypatch.setattr(gpe, "_LIB", s.lib)
    s.limits()
    yield s
    s.limits()
