"""The library's host side on a HIP runtime of host memory
(host_runtime/host_runtime.hip), which runs no kernel but can refuse launches
and allocations: what a draw leaves behind when one of its steps fails, which
forms and splits are taken, and the grids and queues of the kernels."""
import ctypes
import glob
import os
import re
import subprocess

import numpy as np
import pytest

from skity_amd import abi, build, device, presizer
from skity_amd.canvas import Canvas, Paint, Path

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "host_runtime", "host_runtime.hip")
LIB = os.path.join(HERE, "host_runtime", "libskity_host_runtime.so")
ERROR_DEVICE, ERROR_OUT_OF_DEVICE_MEMORY = -6, -7
OBJS = [os.path.join(build.HERE, "_build", u.replace(".hip", ".o")) for u in build.HIP_UNITS]


@pytest.fixture(scope="module")
def runtime():
    if not os.path.exists(build.HIPCC):
        pytest.skip("hipcc not available")
    units = glob.glob(os.path.join(build.HERE, "csrc", "*.h*"))
    if not all(map(os.path.exists, OBJS)) or \
            min(map(os.path.getmtime, OBJS)) < max(map(os.path.getmtime, units)):
        build.build_hip()
    if not os.path.exists(LIB) or \
            os.path.getmtime(LIB) < max(map(os.path.getmtime, OBJS + [SRC])):
        obj = LIB + ".o"
        subprocess.run([build.HIPCC, "--cuda-host-only", "-O1", "-std=c++17", "-fPIC",
                        "-DHIPR_TEMPLATES_ONLY", "-Wno-unused-value", "-Wno-unused-result",
                        "-c", "-o", obj, SRC], check=True)
        subprocess.run(["g++", "-shared", "-o", LIB + ".tmp", *OBJS, obj, "-Wl,-Bsymbolic"],
                       check=True)
        os.remove(obj)
        os.replace(LIB + ".tmp", LIB)
    real, real_load = device._lib, abi.load
    L = ctypes.CDLL(LIB)
    L.test_log.restype = ctypes.c_char_p
    L.test_limit_malloc.argtypes = [ctypes.c_int64]
    for fn in (L.test_unfinished, L.test_copied):
        fn.restype = ctypes.c_int64
    device._lib, abi.load = None, lambda name: L
    device.lib()
    abi.load = real_load
    yield L
    device._lib = real


class Frame:
    """`n` draws on a canvas of `side` pixels whose flattened bounds, edge
    counts and active-edge bounds are the given ones, in turn."""

    def __init__(self, L, side, n, ltrb, edges, bound):
        L.test_reset()
        a = [np.ascontiguousarray(ltrb, np.float32), np.ascontiguousarray(edges, np.int32),
             np.ascontiguousarray(bound, np.int32)]
        L.test_set_frame(len(a[1]), *(ctypes.c_void_p(x.ctypes.data) for x in a))
        self.L = L
        self.ctx = device.Context(0)
        presizer.install(self.ctx, *presizer.load())
        c = Canvas(side, side)
        for i in range(n):
            c.draw_path(Path().move_to(1, 1).line_to(9, 2).line_to(3, 8).close(),
                        Paint((0.5, 0.1, 0.1, 1.0)))
        self.scene = c.scene()
        self.surf = device.Surface(self.ctx, side, side)
        self.prep = device.Prepared(self.ctx, self.scene.scene)

    def launches(self):
        return self.L.test_log().decode().splitlines()

    def kernels(self):
        """Names and grids, in launch order."""
        return [k.rsplit(" ", 1)[0] for k in self.launches()]

    def queues(self):
        return {int(k.rsplit(" ", 1)[1]) for k in self.launches()}

    def draw(self, limit=-1, **kw):
        """The kernels of a draw that may allocate `limit` bytes at a time."""
        self.L.test_reset()
        self.L.test_limit_malloc(limit)
        self.surf.draw(self.prep, **kw)
        return self.kernels()

    def close(self):
        self.surf.close()
        self.prep.close()
        self.ctx.close()


def tiers(L):
    """Draws of every width of the walk (1 .. 64 slots), some tall: a plan of
    schedule passes and writes on all streams."""
    side = 2048
    tall, low = (0, 0, 300, 1900), (10, 10, 500, 90)
    bound = [40, 40, 100, 200, 200, 400, 900, 1500, 3000]
    ltrb = [low, tall, low, tall, low, tall, tall, low, tall]
    return Frame(L, side, len(bound), ltrb, [200] * 5 + [4000] * 4, bound)


@pytest.mark.parametrize("kw", [dict(mode=abi.MODE_EXACT), dict(mode=abi.MODE_EXACT, band_rows=64),
                                dict(mode=abi.MODE_LEARNED),
                                dict(mode=abi.MODE_LEARNED, flags=abi.FLAG_PERSISTENT)])
def test_a_plan_that_fails_leaves_nothing_running(runtime, kw):
    """Whichever walk launch of a draw is refused, every kernel launched before
    it has been waited for when the draw returns: the next draw takes their
    buffers."""
    f = tiers(runtime)
    names = f.draw(**kw)
    walks = sum("WalkKernel" in k for k in names)
    assert walks >= 8
    assert runtime.test_unfinished() == 0
    for at in range(walks):
        runtime.test_reset()
        runtime.test_fail_launch(b"WalkKernel", at)
        with pytest.raises(device.HiprError) as e:
            f.surf.draw(f.prep, **kw)
        assert e.value.code == ERROR_DEVICE
        assert runtime.test_unfinished() == 0, at
        assert f.draw(**kw) == names
    f.close()


COUNT, WRITE, SCHEDULE = "0", "1", "2"


def walk_modes(names):
    return {m.group(1) for m in (re.search(r"WalkKernelILi\d+ELi(\d)E", k) for k in names) if m}


def test_planes_are_counted_where_they_cannot_be_reserved(runtime):
    """64 draws over all of 2048 x 2048 could use 512 MiB of planes.  An exact
    draw that cannot reserve them counts them, as one with bands of its own
    does, and reserves them again once it can."""
    f = Frame(runtime, 2048, 64, [(0, 0, 2048, 2048)], [50], [40])
    assert walk_modes(f.draw(limit=64 << 20)) == {COUNT, WRITE}
    assert COUNT not in walk_modes(f.draw())
    assert COUNT not in walk_modes(f.draw(limit=64 << 20))  # kept from the last draw
    assert runtime.test_copied() == 0
    f.close()


def test_bands_are_given_up_where_their_states_cannot_be_reserved(runtime):
    """Two draws of 4,000 edges and 32 bands hold 16 MiB of edge states, and
    512 KiB without bands."""
    f = Frame(runtime, 2048, 2, [(0, 0, 64, 1900)], [4000], [40])
    assert walk_modes(f.draw(limit=8 << 20)) == {WRITE}
    assert walk_modes(f.draw()) == {SCHEDULE, WRITE}
    f.close()


@pytest.mark.parametrize("mode", [abi.MODE_EXACT, abi.MODE_LEARNED])
def test_a_draw_without_memory_is_refused_alone(runtime, mode):
    """Whatever allocation is refused, the draw says so, and the next one is
    not told of it."""
    f = tiers(runtime)
    names = f.draw(mode=mode)
    f.close()
    for limit in (100, 4 << 10, 16 << 10, 64 << 10, 256 << 10):
        f = tiers(runtime)
        with pytest.raises(device.HiprError) as e:
            f.draw(limit=limit, mode=mode)
        assert e.value.code == ERROR_OUT_OF_DEVICE_MEMORY, limit
        assert runtime.test_unfinished() == 0
        assert f.draw(mode=mode) == names
        f.close()


def test_growing_planes_are_not_copied(runtime):
    """A larger frame on the same context takes larger planes; nothing of the
    last frame's is kept."""
    small = Frame(runtime, 2048, 4, [(0, 0, 300, 300)], [50], [40])
    for mode in (abi.MODE_EXACT, abi.MODE_LEARNED):
        for side in (300, 900, 2000):
            runtime.test_set_frame(1, *(x.ctypes.data_as(ctypes.c_void_p) for x in (
                np.array([0, 0, side, side], np.float32), np.array([50], np.int32),
                np.array([40], np.int32))))
            small.draw(mode=mode)
            assert runtime.test_copied() == 0, (mode, side)
    small.close()


def batch_of(f):
    b = device.Batch(f.ctx)
    b.add(f.surf, f.prep)
    return b


def batch_draw(f, b, **kw):
    f.L.test_reset()
    b.draw(**kw)
    return f.kernels()


def test_the_default_split_is_tried_first(runtime):
    """Device time is the number of kernels here.  The exact form is fastest
    without a count pass, which every other split asks for; where nothing is
    banded all splits tie, and the default, the first, is kept."""
    f = tiers(runtime)
    b = batch_of(f)
    names = batch_draw(f, b)
    assert b.autotune(abi.MODE_EXACT, repeats=1) == (0, 0, 0)
    assert batch_draw(f, b) == names
    b.close()
    f.close()
    f = Frame(runtime, 256, 4, [(0, 0, 90, 90)], [50], [40])
    b = batch_of(f)
    for mode in (abi.MODE_EXACT, abi.MODE_LEARNED):
        assert b.autotune(mode, repeats=1) == (0, 0, 0)
    b.close()
    f.close()


def test_splits_are_tried_where_planes_are_counted(runtime):
    """More planes than are ever reserved: the default counts them too, and one
    band per path saves nothing but may be chosen."""
    f = Frame(runtime, 2048, 520, [(0, 0, 2048, 2048)], [50], [40])
    b = batch_of(f)
    assert COUNT in walk_modes(batch_draw(f, b))
    runtime.test_reset()
    assert b.autotune(abi.MODE_EXACT, repeats=1) == (0, 0, 0)
    draws = sum("JobTileRangeKernel" in k for k in f.kernels())
    assert draws >= 2 * 2 * 4  # two draws each of four splits, launched in two ways
    b.close()
    f.close()


def test_a_split_is_used_by_the_form_it_was_tuned_for(runtime):
    """A split tuned for learned draws would make exact ones count.  Tuning
    again does not start from the split found before."""
    f = tiers(runtime)
    b = batch_of(f)
    exact = batch_draw(f, b)
    split = b.autotune(abi.MODE_LEARNED, repeats=1)
    assert split[0] < 0  # no schedule pass: the fewest kernels
    tuned = batch_draw(f, b, mode=abi.MODE_LEARNED)
    assert walk_modes(tuned) == {WRITE}
    assert batch_draw(f, b) == exact
    assert b.autotune(abi.MODE_LEARNED, repeats=1) == split
    b.set_split(64, 0)  # a caller's own split holds for every form
    assert COUNT in walk_modes(batch_draw(f, b))
    b.close()
    f.close()


@pytest.mark.parametrize("mode", [abi.MODE_EXACT, abi.MODE_LEARNED])
def test_persistent_walks_fill_the_device(runtime, mode):
    """Every walk of the persistent form has a workgroup per item, up to the
    2,048 that fit the device at once here, whatever the frame's other walks."""
    def grids(names):
        return [int(k.split()[1]) for k in names if "WalkKernel" in k]

    f = Frame(runtime, 2048, 300, [(0, 0, 300, 1900)] * 2 + [(9, 9, 90, 50)] * 3,
              [300] * 5, [40, 300, 20, 100, 600])
    plain = grids(f.draw(mode=mode))
    assert len(plain) >= 5 and max(plain) < 2048
    assert grids(f.draw(mode=mode, flags=abi.FLAG_PERSISTENT)) == plain
    f.close()
    f = Frame(runtime, 2048, 3000, [(9, 9, 90, 50)], [300], [20])
    assert grids(f.draw(mode=mode)) == [3000]
    assert grids(f.draw(mode=mode, flags=abi.FLAG_PERSISTENT)) == [2048]
    f.close()


def test_contexts_take_different_queues(runtime):
    """Frames of one walk kernel run on their context's main stream alone; four
    contexts use the four hardware queues."""
    frames = [Frame(runtime, 256, 4, [(0, 0, 90, 90)], [50], [40]) for _ in range(4)]
    used = []
    for f in frames:
        f.draw()
        used.append(f.queues())
        f.close()
    assert all(len(q) == 1 for q in used)
    assert set.union(*used) == {0, 1, 2, 3}
