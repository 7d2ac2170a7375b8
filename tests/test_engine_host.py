"""CPU tests of the engine's host code: csrc/atmo_engine.cpp and the launchers of
csrc/atmo_kernels.hip, compiled for the host only and linked with a host-side HIP
runtime (native/fake_hip.cpp) that can refuse memory and launches.  Kernels do not run."""
import ctypes
import os
import re
import shutil
import subprocess

import pytest

from prolandatmo import lib as L
from prolandatmo.params import FLAG_NO_AUTOTUNE, AtmoParams, earth, options, with_res

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "proland-4.0_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
OK, DEVICE, OOM = 0, 2, 3


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("engine_host")
    host = [HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-w", "-x", "hip", "-c"]
    objs = []
    native = os.path.join(REPO, "tests", "native")
    for src in (os.path.join(CSRC, "atmo_engine.cpp"), os.path.join(CSRC, "atmo_kernels.hip"),
                os.path.join(native, "host_calls.cpp")):
        name = os.path.basename(src).split(".")[0]
        objs.append(str(d / (name + ".o")))
        subprocess.check_call(host + ["-cuid=" + name, src, "-o", objs[-1]])
    objs.append(str(d / "fake.o"))
    subprocess.check_call(["g++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-O1", "-std=c++17", "-fPIC", "-w", "-c",
                           os.path.join(native, "fake_hip.cpp"), "-o", objs[-1]])
    so = str(d / "engine_host.so")
    device_code = set(re.findall(r"__hip_fatbin_\w+", subprocess.check_output(["nm"] + objs, text=True)))
    # every symbol bound inside the library: the process may hold the real runtime too
    subprocess.check_call(["g++", "-shared", "-Wl,-Bsymbolic", "-o", so] + objs +
                          ["-Wl,--defsym=%s=fake_fatbin" % s for s in sorted(device_code)])
    lib = ctypes.CDLL(so)
    for name, (res, args) in L.SIGNATURES.items():
        if hasattr(lib, name):
            getattr(lib, name).restype, getattr(lib, name).argtypes = res, args
    lib.fake_memory_limit.argtypes = [ctypes.c_size_t]
    lib.fake_in_use.restype = ctypes.c_size_t
    return lib


class Engine:
    """The C ABI's engine on the host runtime; outputs are addresses that nothing reads."""

    def __init__(self, lib):
        self.lib, self.h = lib, ctypes.c_void_p()
        lib.fake_reset()
        assert lib.atmo_engine_create(ctypes.byref(self.h), 0) == OK

    def __enter__(self):
        return self

    def __exit__(self, *a):
        self.lib.fake_reset()
        self.lib.atmo_engine_destroy(self.h)

    def precompute(self, p, o, stream=1):
        sets = (AtmoParams * 1)(p)
        out = (L.AtmoTables * 1)(L.AtmoTables(0x1000, 0x2000, 0x3000))
        return self.lib.atmo_engine_precompute(self.h, sets, 1, ctypes.byref(o), out, ctypes.c_void_p(0x100 * stream))


def small(k=0):
    p = with_res(earth(), 4, 8, 4, 2)
    p.HR = 8.0 + 0.125 * k
    return p


def plain(orders=4):
    return options(orders=orders, flags=FLAG_NO_AUTOTUNE)


def test_precompute_without_room_for_the_view_samples(host):
    """A set whose work memory fits only without the table of view-ray samples and the
    theta rows is computed without them: the refused allocation leaves no error behind."""
    p, o = small(), plain()
    with Engine(host) as e:
        assert e.precompute(p, o) == OK
        full, launches = host.fake_in_use(), host.fake_launch_count()
    with Engine(host) as e:
        host.fake_memory_limit(full - 1024)
        assert e.precompute(p, o) == OK, host.atmo_last_error()
        assert host.fake_in_use() < full - 1024
        assert host.fake_launch_count() == launches - 1   # all but the view samples' kernel
        assert host.fake_pending() == 0


def test_precompute_after_one_that_did_not_fit(host):
    with Engine(host) as e:
        host.fake_memory_limit(1 << 16)
        assert e.precompute(small(), plain()) == OOM
        host.fake_memory_limit(1 << 40)
        assert e.precompute(small(1), plain()) == OK, host.atmo_last_error()


def test_work_memory_of_a_run_that_failed_is_not_handed_over(host):
    """A plan whose launches fail part way has no event behind the ones that went out:
    the next plan, on another stream, waits for the device instead of for an event of
    the plan two before."""
    with Engine(host) as e:
        for k in range(2):
            assert e.precompute(small(k), plain()) == OK
        host.fake_fail_launch(5)
        assert e.precompute(small(2), plain()) == DEVICE
        assert e.precompute(small(3), plain(), stream=2) == OK, host.atmo_last_error()
        assert e.precompute(small(4), plain(), stream=2) == OK
        assert host.fake_stale_waits() == 0


@pytest.mark.parametrize("after", [1, 2, 3])
def test_work_memory_is_handed_over_behind_the_last_run(host, after):
    """Plans that run once on alternating streams, then one that runs `after` times."""
    with Engine(host) as e:
        for k in range(4):
            assert e.precompute(small(k), plain(), stream=1 + k % 2) == OK
        for _ in range(after):
            assert e.precompute(small(4), plain(), stream=1) == OK
        assert e.precompute(small(5), plain(), stream=1) == OK
        assert host.fake_stale_waits() == 0
        assert host.fake_pending() == 0


def launches(lib):
    """(grid, block, dynamic LDS) of every launch so far."""
    out = []
    for i in range(lib.fake_launch_count()):
        grid, block, lds = (ctypes.c_uint * 3)(), ctypes.c_uint(), ctypes.c_size_t()
        lib.fake_launch(i, grid, ctypes.byref(block), ctypes.byref(lds))
        out.append((tuple(grid), block.value, lds.value))
    return out


@pytest.mark.parametrize("RR,RMUS,SW,SH,NS,NI", [
    (32, 32, 64, 16, 16, 32), (2, 2, 2, 2, 1, 2), (64, 64, 64, 16, 32, 32),
    # the most layers (a table of 2^27 texels) and rows that are accepted, with the most directions
    (1 << 23, 2, 64, 16, 128, 32), (1 << 23, 2, 2, 1 << 23, 128, 256)])
def test_theta_table_workgroups(host, RR, RMUS, SW, SH, NS, NI):
    """Items of the theta tables: ground transmittances and dJ rows, dE rows, columns, the
    first three each padded to a wave."""
    pad = lambda n: (n + 63) // 64 * 64
    items = 2 * pad(RR * NS) + pad(SH * (NI // 2)) + SW + RMUS
    assert host.call_theta_workgroups(RR, RMUS, SW, SH, NS, NI) == (items + 255) // 256


@pytest.mark.parametrize("nsets,wpt,nview", [
    (1, 11, 51), (3, 0, 7), (1, 1 << 23, 1 << 21), (2, 12_600_000, 3), (1, 2, 5_000_000), (40_000, 1000, 1), (3, 0, 3_000_000)])
def test_geometry_launches_stay_below_2_to_32_threads(host, nsets, wpt, nview):
    host.fake_reset()
    assert host.call_launch_geometry(nsets, wpt, nview) == 0
    total = 0
    for grid, block, _ in launches(host):
        assert block == 256 and grid[1] == grid[2] == 1
        assert grid[0] * block < 1 << 32
        total += grid[0]
    assert total == nsets * wpt + 16 * nview


@pytest.mark.parametrize("linear", [0, 1])
def test_inscatter1_shapes_cover_the_row_and_fit_the_lds(host, linear):
    """Every row length and T widths from the least to past the staged columns: a staged
    launch covers the row's texels and T's columns, and takes at most 64 KB of dynamic LDS."""
    largest = 0
    for W4 in range(4, 1025):
        for TW in (2, 63, 64, 128, 256, 257, 512, 1000, 1024, 1025, 1403, 1404, 1536, 1537, 2048, 2049, 4096):
            shape = (ctypes.c_int * 3)()
            host.fake_reset()
            assert host.call_inscatter1(W4, TW, linear, shape) == 0
            (grid, block, lds), = launches(host)
            texels, columns, threads = shape
            assert block == threads <= 512 and lds <= 64 * 1024
            assert texels == 0 or (texels * threads >= W4 and columns * threads >= TW)
            largest = max(largest, lds)
    assert largest == (32 * (4 * 384 + 1) + (0 if linear else 8 * 1536))
