"""The library's host side on a HIP runtime in host memory (fake_hip.cpp:
allocations can be made to fail, kernels do not run): what it allocates and
launches, and that a call that runs out of memory returns an error and leaves
nothing behind that a later call would hand to a kernel. CPU only."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PREAMBLE = """
import ctypes, sys
sys.path.insert(0, {root!r})
F = ctypes.CDLL({fake!r}, ctypes.RTLD_GLOBAL)  # before librgrt.so: its symbols come first
F.fake_log.restype = ctypes.c_char_p
import numpy as np
from raygun_amd import rgrt
from raygun_amd.records import INSTANCE, RAY, UBO, VERTEX
from raygun_amd.rgrt import Context, RgrtError

def log():
    return F.fake_log().decode().split("\\n")

def launches(name):
    return [l.split() for l in log() if l.startswith("launch") and name in l]

def allocations(name="hipMalloc"):
    return [int(l.split()[1]) for l in log() if l.startswith(name + " ")]

def fail(name, nth=1):
    F.fake_fail(name.encode(), nth)

def raises(f):
    try:
        f()
    except RgrtError as e:
        return str(e)
    raise AssertionError("no error")

def one_triangle(ctx):
    v = np.zeros(3, VERTEX)
    v["position"] = [[0, 0, 0], [1, 0, 0], [0, 1, 0]]
    ctx.upload_geometry(v, np.arange(3))
    inst = np.zeros(1, INSTANCE)
    inst["blas"] = ctx.build_blas(0, 0, 1, 3)
    inst["transform"] = [1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0]
    inst["mask"] = 0xFF
    ctx.build_tlas(inst)
    return inst
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    fake = str(tmp_path_factory.mktemp("fake_hip") / "fake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "fake_hip.cpp"), "-o", fake], check=True)

    def go(body):
        r = subprocess.run([sys.executable, "-c", PREAMBLE.format(root=ROOT, fake=fake) + body], capture_output=True, text=True,
                           timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr

    return go


def test_pinned_ray_memory_without_a_device_address(run):
    """The pinned buffer of small host queries is there with its device
    address or not at all: no query runs on a null one."""
    run("""
fail("hipHostGetDevicePointer")
try:
    ctx = Context(16, 16)
except RgrtError:
    ctx = Context(16, 16)
else:
    one_triangle(ctx)
    raises(lambda: ctx.trace_rays(np.zeros(1, RAY)))
    log()
    ctx.trace_rays(np.zeros(1, RAY))
    assert allocations("hipHostMalloc"), "a query after the failed one ran without the buffer"
one_triangle(ctx)
log()
ctx.trace_rays(np.zeros(4, RAY))
assert len(launches("k_trace_rays")) == 1
""")


@pytest.mark.parametrize("rays", [1, 5000])
def test_ray_queries_without_images(run, rays):
    """A context of size 0 x 0 answers ray queries: the error word of the
    traversal is there without a frame's counters."""
    run(f"""
ctx = Context(0, 0)
one_triangle(ctx)
assert len(ctx.trace_rays(np.zeros({rays}, RAY))) == {rays}
""")


def test_first_frame_of_several_samples_keeps_the_queue_of_rays_ahead(run):
    """The slot arrays grow with the samples; the queue of rays ahead has one
    size from 300,000 slots on and is not allocated again."""
    run("""
ctx = Context(800, 600)
queue = 300000 * 2 * 7 * 4
assert queue in allocations()
inst = one_triangle(ctx)
ubo = np.zeros((), UBO)
ubo["numSamples"], ubo["maxRecursions"] = 3, 1
log()
ctx.frame(ubo, inst)
grown = allocations()
assert 3 * 800 * 600 * 10 * 4 in grown and queue not in grown, grown
""")


GROWING = {
    # (a call, the same on something larger, the allocation that fails)
    "rays": ("ctx.trace_rays(np.zeros(5000, RAY))", "ctx.trace_rays(np.zeros(9000, RAY))", "hipMalloc", 2),
    "slots": ("frame(1)", "frame(3)", "hipMalloc", 2),
    "sample records": ("frame(2)", "frame(3)", "hipMalloc", 6),
    "pass counts": ("ctx.set_sample_groups(1); frame(1)", "frame(3, 7)", "hipHostMalloc", 1),
    "images": ("ctx.resize(16, 16); frame(1)", "ctx.resize(24, 24)", "hipMalloc", 3),
    "8-bit image": ("ctx.resize(16, 16); ctx.read_image_rgba8()", "ctx.resize(24, 24); log(); fail('hipMalloc'); ctx.read_image_rgba8()",
                    "", 0),
    "instances": ("ctx.build_tlas(inst); ctx.trace_rays(np.zeros(1, RAY))", "ctx.build_tlas(np.repeat(inst, 100))", "hipMalloc", 3),
    "stack spill": ("ctx.set_tuning(drainBlocksPerCU=4)", "ctx.set_tuning(drainBlocksPerCU=32)", "hipMalloc", 1),
    "network": ("den.infer(np.zeros((1, 16, 16, 16)))", "den.infer(np.zeros((1, 64, 64, 16)))", "hipMalloc", 1),
}


@pytest.mark.parametrize("what", GROWING)
def test_a_buffer_that_could_not_grow_is_allocated_by_the_next_call(run, what):
    """What was freed to make room is not taken for what it was: the smaller
    call allocates again and succeeds."""
    small, large, function, nth = GROWING[what]
    run(f"""
ctx = Context(16, 16)
inst = one_triangle(ctx)
den = rgrt.Denoiser(ctx)
den.set_params(den.get_params())

def frame(samples, recursions=1):
    ubo = np.zeros((), UBO)
    ubo["numSamples"], ubo["maxRecursions"] = samples, recursions
    ctx.frame(ubo, inst)

def small():
    {small}

def large():
    {large}

small()
if {function!r}:
    fail({function!r}, {nth})
assert "out of memory" in raises(large)
if {what!r} == "instances":
    assert "no TLAS" in raises(lambda: ctx.trace_rays(np.zeros(1, RAY)))
if {what!r} == "images":
    assert "zero-sized" in raises(lambda: frame(1))
log()
small()
l = log()
assert any(x.startswith("hipMalloc") or x.startswith("hipHostMalloc") for x in l), l
log()
small()
assert not allocations()
""")


@pytest.mark.parametrize("holds", [3, 5, 40])
def test_launch_shape_reads_back_as_launched(run, holds):
    """traceBlocksPerCU beyond what a CU holds is what it holds, in the grid
    and in what rgrt_get_tuning says."""
    run(f"""
F.fake_occupancy({holds})
ctx = Context(16, 16)
inst = one_triangle(ctx)
ubo = np.zeros((), UBO)
ubo["numSamples"], ubo["maxRecursions"] = 1, 1
assert ctx.tuning()["traceBlocksPerCU"] == min(5, {holds})
for blocks in (1, 4, 8, 32):
    ctx.set_tuning(traceBlocksPerCU=blocks)
    assert ctx.tuning()["traceBlocksPerCU"] == min(blocks, {holds})
    log()
    ctx.frame(ubo, inst)
    grids = [int(l[2]) for l in launches("k_trace_queue")]
    assert grids and all(g == 2 * min(blocks, {holds}) for g in grids), grids  # two CUs
""")
