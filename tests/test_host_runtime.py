"""The library's host code over a HIP runtime on the CPU (native/hip_stub.cpp): which kernels it
launches, on which device it makes its events, what it does with errors.  Each case runs in a process
of its own, where the stub is loaded ahead of the library."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)

PRELUDE = """
import ctypes, json, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import numpy as np
import activemodelbplus.integrator as amb
from activemodelbplus import tuning
stub.stub_launch.restype = ctypes.c_char_p

def launches():
    out = []
    for i in range(stub.stub_launches()):
        b, t, l = ctypes.c_uint(), ctypes.c_uint(), ctypes.c_size_t()
        name = stub.stub_launch(i, ctypes.byref(b), ctypes.byref(t), ctypes.byref(l)).decode()
        out.append((name, b.value, t.value, l.value))
    return out

def steps():  # names of the step kernels launched since the last call
    out = [name for name, *_ in launches() if "step_kernel" in name or "march_kernel" in name]
    stub.stub_clear()
    return out

def model(T):
    return amb.Model(-0.25, 0, 0.25, 1, 0.5, -1, T)

stencil = amb.Stencil(5e-3, 1, 1)
"""


@pytest.fixture(scope="module")
def on_stub(tmp_path_factory):
    """on_stub(code): what the code, run on the stub, prints as its last line (JSON)."""
    lib = str(tmp_path_factory.mktemp("hip") / "libhipstub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "native", "hip_stub.cpp"), "-o", lib], check=True)

    def run(code):
        res = subprocess.run([sys.executable, "-c", PRELUDE + code, lib, os.path.join(REPO, "active-model-bplus_amd")],
                             capture_output=True, text=True, timeout=120)
        assert res.returncode == 0, res.stderr[-2000:]
        return json.loads(res.stdout.strip().splitlines()[-1])

    return run


@pytest.mark.parametrize("precision", [32, 64])
def test_ensemble_autotune_times_the_kernels_that_run(on_stub, precision):
    """Members with noise on columns that do and do not split into fours have kernels of their own
    (noise modes 1 and 3); the autotuner times the one that each member runs."""
    timed, ran = on_stub(f"""
fields = [np.zeros((200, 201)), np.zeros((200, 200)), np.zeros((200, 199))]
ens = amb.Ensemble(fields, stencil, [model(0.05), model(0.05), model(0.0)], [1, 2, 3], precision={precision})
assert ens.resident_count == 0
steps()
ens.autotune(1)
timed = steps()
ens.run(1)
mode = lambda names: sorted(set(n.split("ELi")[3][0] for n in names))
print(json.dumps([mode(timed), mode(steps())]))
""")
    assert ran == ["0", "1", "3"]
    assert timed == ran


@pytest.mark.parametrize("precision", [32, 64])
def test_getters_with_another_device_current(on_stub, precision):
    """A field of more than one staging piece is read while another GPU is current, and that GPU
    stays current."""
    ok = on_stub(f"""
n = (400, 512)
phi = np.arange(n[0] * n[1], dtype=np.float64).reshape(n)
sim = amb.Integrator(phi, stencil, model(0), precision={precision})
ens = amb.Ensemble([phi[:7], phi], stencil, [model(0)] * 2, [1, 2], precision={precision})
stub.hipSetDevice(1)
ok = [bool((sim.field == phi).all()), bool((ens.field(1) == phi).all())]
d = ctypes.c_int(-1)
stub.hipGetDevice(ctypes.byref(d))
print(json.dumps(ok + [d.value]))
""")
    assert ok == [True, True, 1]


def test_getters_of_one_field_take_turns(on_stub):
    """Observables of one field share their device buffer: from the launch of an observable to the
    copy of its last value no other thread's getter launches or copies anything."""
    order = on_stub("""
import threading
n = (1024, 512)  # four pieces a component
lib = ctypes.CDLL(sys.argv[2] + "/lib/libamb.so")
h = ctypes.c_void_p()
class Options(ctypes.Structure):
    _fields_ = [("precision", ctypes.c_int), ("seed", ctypes.c_uint64), ("timestep", ctypes.c_int64), ("tile", ctypes.c_int)]
three, seven = (ctypes.c_double * 3)(5e-3, 1, 1), (ctypes.c_double * 7)(-0.25, 0, 0.25, 1, 0.5, -1, 0.05)
phi = np.zeros(n)
opt = Options(32, 1, 0, 0)
ptr = lambda a: ctypes.c_void_p(a.ctypes.data)
assert lib.amb_create(ptr(phi), ctypes.c_int64(n[0]), ctypes.c_int64(n[1]), three, seven, ctypes.byref(opt), ctypes.byref(h)) == 0
stub.stub_clear()
rc = []
def get(which):
    out = np.zeros((2,) + n)
    rc.append(lib.amb_get_observable(h, which, ptr(out)))
threads = [threading.Thread(target=get, args=(w,)) for w in (3, 0, 5, 2)]  # ctypes lets them overlap
for t in threads: t.start()
for t in threads: t.join()
assert rc == [0] * 4
buf = (ctypes.c_ulong * 1000)()
k = stub.stub_order(buf, 1000)
print(json.dumps(list(buf[:k])))
""")
    threads = [x // 2 for x in order]
    assert len(set(threads)) == 4
    assert sum(a != b for a, b in zip(threads, threads[1:])) == 3, threads


LARGE = """
shape, precision, T = {shape}, {precision}, {T}
phi = np.zeros(shape)
make = lambda tile=0: amb.Integrator(phi, stencil, model(T), seed=1, precision=precision, tile=tile)
shapes = [tuple(s) for s in amb.tile_shapes(precision)]
square = shapes.index((32, 32, 512))
def ran(sim):  # "strips" or the shape of the step's tiles
    stub.stub_clear()
    sim.run(1)
    (name,) = steps()
    return "strips" if "march" in name else tuple(int(x.split("E")[0]) for x in name.split("Li")[1:4])
"""
FIELDS = pytest.mark.parametrize("shape,precision,T", [((2050, 2050), 32, 0.05), ((2304, 2304), 32, 0.0),
                                                       ((1800, 1801), 64, 0.05), ((2304, 2304), 64, 0.0)])


@FIELDS
def test_a_chosen_shape_is_the_shape_that_runs(on_stub, shape, precision, T):
    """Fields large enough for strips run in them when no tile was chosen; every shape can be chosen,
    by the option and by set_tile."""
    out = on_stub(LARGE.format(shape=shape, precision=precision, T=T) + """
by_option = [ran(make(t + 1)) for t in range(len(shapes))]
sim = make()
first = ran(sim)
by_set = []
for t in range(len(shapes)):
    sim.set_tile(t)
    by_set.append(ran(sim))
print(json.dumps([first, by_option == shapes, by_set == shapes]))
""")
    assert out == ["strips", True, True]


@FIELDS
def test_autotune_times_strips_beside_the_shapes(on_stub, shape, precision, T):
    """Whichever is fastest runs afterwards, also in new fields of that size and where the table is
    asked first; the index returned is a shape's either way."""
    out = on_stub(LARGE.format(shape=shape, precision=precision, T=T) + """
out = []
for fast, want in (("march_kernel", "strips"), ("Li32ELi32ELi512E", shapes[square]), ("Li64ELi16ELi256E", (64, 16, 256))):
    tuning.clear()
    stub.stub_fast(fast.encode())
    sim = make()
    best = sim.autotune(1)
    timed = len(set(steps()))
    assert timed == len(shapes) + 1 and 0 <= best < len(shapes)
    assert amb.tuning_get(precision, shape[0], shape[1], T > 0) == best
    again = make(3)
    assert again.autotune(1, cached=True) == best and not steps()
    out.append([ran(sim) == want, ran(make()) == want, ran(again) == want])
print(json.dumps(out))
""")
    assert out == [[True] * 3] * 3


@FIELDS
def test_ensemble_timing_leaves_single_fields_their_strips(on_stub, shape, precision, T):
    """An ensemble's timing, and a file of one that says nothing of strips, neither take them from
    single fields of that size nor replace what a single field's timing found."""
    out = on_stub(LARGE.format(shape=shape, precision=precision, T=T) + """
import os, tempfile
path = os.path.join(tempfile.mkdtemp(), "tiles.json")
key = precision, shape[0], shape[1], T > 0
stub.stub_fast(b"Li64ELi16ELi256E")
ens = lambda: amb.Ensemble([phi], stencil, [model(T)], [1], precision=precision)
tile = ens().autotune(1)[0]
out = [shapes[tile] == (64, 16, 256), amb.tuning_get(*key) == tile, ens().tiles[0] == tile, ran(make()) == "strips"]
tuning.save(path)
tuning.clear()
tuning.load(path)
out += [ens().tiles[0] == tile, ran(make()) == "strips"]
data = json.load(open(path))
for e in data["entries"]:
    del e["timed"]  # a file of before
json.dump(data, open(path, "w"))
tuning.clear()
assert tuning.load(path) == 1
out += [ens().tiles[0] == tile, ran(make()) == "strips"]
steps()
make().autotune(1, cached=True)  # no entry that would do: times
out += [len(set(steps())) == len(shapes) + 1, ran(make()) == (64, 16, 256)]
for fast, runs in (("march_kernel", "strips"), ("Li32ELi16ELi256E", (32, 16, 256))):
    stub.stub_fast(fast.encode())
    make().autotune(1)
    kept = amb.tuning_get(*key)
    stub.stub_fast(b"Li64ELi16ELi256E")
    ens().autotune(1)
    out += [amb.tuning_get(*key) == kept, ran(make()) == runs]
    tuning.save(path)
    tuning.clear()
    tuning.load(path)
    out += [amb.tuning_get(*key) == kept, ran(make()) == runs]
amb.tuning_set(*key, 1)
print(json.dumps(out + [ran(make()) == shapes[1]]))
""")
    assert out == [True] * len(out)


@pytest.mark.parametrize("precision", [32, 64])
def test_step_shape_names_what_runs(on_stub, precision):
    """At every size of the library's choice, with a chosen tile, and with an explicit noise buffer
    (which strips do not take)."""
    out = on_stub(LARGE.format(shape=(64, 64), precision=precision, T=0.05) + """
import math
out, seen = [], set()
for shape, T in [((64, 64), 0.0), ((256, 256), 0.05), ((512, 512), 0.0), ((704, 704), 0.05), ((1088, 1090), 0.0),
                 ((1088, 1088), 0.05), ((2050, 2049), 0.05), ((2304, 2304), 0.0)]:
    for tile in (0, 1, 3):
        sim = amb.Integrator(np.zeros(shape), stencil, model(T), seed=1, precision=precision, tile=tile)
        for noise in (False, True):
            if noise:
                sim.set_noise(np.zeros((1, 2) + shape))
            cols, rows, threads, strips = sim.step_shape
            seen.add("strips" if strips else (cols, rows, threads))
            stub.stub_clear()
            sim.run(1)
            ((name, blocks, nt, _),) = [l for l in launches() if "step_kernel" in l[0] or "march_kernel" in l[0]]
            work = math.ceil(shape[0] / rows) * math.ceil(shape[1] / cols)
            out.append(strips == ("march" in name) and nt == threads and work <= blocks)
            out.append(strips or f"Li{cols}ELi{rows}ELi{threads}E" in name)
            out.append(not (strips and (noise or tile)))
print(json.dumps([out, "strips" in seen, (32, 16, 512) in seen, (32, 32, 512) in seen]))
""")
    assert out == [[True] * len(out[0]), True, True, True]


def test_bench_reads_the_profile_of_what_runs(on_stub):
    """The benchmark's traffic and instruction counts are those of the default run's strips, and a
    chosen shape does not get them."""
    out = on_stub(f"""
sys.path.insert(0, {REPO!r})
import bench
out = []
for key in ("c3", "c3x8192"):
    w = bench.WORKLOADS[key]
    make = lambda tile: amb.Integrator(np.zeros((w["n"], w["n"])), amb.Stencil(*w["stencil"]), amb.Model(*w["model"]),
                                       precision=w["precision"], tile=tile)
    run, chosen = make(0).step_shape[:3], make(10).step_shape[:3]
    out.append(bench.read_traffic(bench.TRAFFIC_PROFILE[key], run) > 8 * w["n"] ** 2)
    out.append(bench.read_traffic(bench.TRAFFIC_PROFILE[key], chosen) is None)
    if key in bench.VALU_PROFILE:
        out.append(bench.read_valu(bench.VALU_PROFILE[key], run) > 0)
print(json.dumps(out))
""")
    assert out == [True] * 5


def test_observable_parts_is_public_and_checked(on_stub):
    """Every amb_ function that the Python module calls is declared in amb.h alone, and a current without a
    place for its second component is refused."""
    csrc = os.path.join(REPO, "active-model-bplus_amd", "csrc")
    assert 'extern "C"' not in open(os.path.join(csrc, "pyintegrator.cpp")).read()
    assert "amb_get_observable_parts(" in open(os.path.join(REPO, "include", "amb.h")).read()
    out = on_stub("""
lib = ctypes.CDLL(sys.argv[2] + "/lib/libamb.so")
ptr = lambda a: ctypes.c_void_p(a.ctypes.data)
phi, h = np.zeros((8, 8)), ctypes.c_void_p()
three, seven = (ctypes.c_double * 3)(5e-3, 1, 1), (ctypes.c_double * 7)(-0.25, 0, 0.25, 1, 0.5, -1, 0.05)
assert lib.amb_create(ptr(phi), ctypes.c_int64(8), ctypes.c_int64(8), three, seven, None, ctypes.byref(h)) == 0
y, x = np.ones((8, 8)), np.ones((8, 8))
rc = [lib.amb_get_observable_parts(h, 3, ptr(y), None), lib.amb_get_observable_parts(h, 0, ptr(y), None),
      lib.amb_get_observable_parts(h, 3, ptr(y), ptr(x))]
print(json.dumps(rc))
""")
    assert out == [1, 0, 0]


def test_strip_tests_run_in_strips(on_stub):
    """Every grid of test_strips_equal_tiles and of the finite check beside it takes strips on a device of
    256 compute units."""
    import test_gpu_step_paths as paths
    (cases,) = [m.args[1] for m in paths.test_strips_equal_tiles.pytestmark if m.name == "parametrize"]
    out = on_stub(f"""
cases = {list(cases) + [(32, (2048, 2050), 0.0)]!r}
print(json.dumps([amb.Integrator(np.zeros(s), stencil, model(T), precision=p).step_shape[3] for p, s, T in cases]))
""")
    assert len(out) >= 9 and all(out)


@pytest.mark.parametrize("precision", [32, 64])
def test_a_small_currents_components_come_in_one_copy(on_stub, precision):
    """To separate arrays (Python's getters) up to 16384 sites, to one array (the C ABI's) at any size
    of one staging piece; the values are the device's."""
    out = on_stub(f"""
lib = ctypes.CDLL(sys.argv[2] + "/lib/libamb.so")
ptr = lambda a: ctypes.c_void_p(a.ctypes.data)
three, seven = (ctypes.c_double * 3)(5e-3, 1, 1), (ctypes.c_double * 7)(-0.25, 0, 0.25, 1, 0.5, -1, 0.05)
class Options(ctypes.Structure):
    _fields_ = [("precision", ctypes.c_int), ("seed", ctypes.c_uint64), ("timestep", ctypes.c_int64), ("tile", ctypes.c_int)]
def copies():
    buf = (ctypes.c_ulong * 1000)()
    k = stub.stub_order(buf, 1000)
    stub.stub_clear()
    return sum(x & 1 for x in buf[:k])
out = []
for ny, nx in ((8, 9), (128, 128), (128, 129), (256, 256)):
    phi, h, opt = np.zeros((ny, nx)), ctypes.c_void_p(), Options({precision}, 1, 0, 0)
    assert lib.amb_create(ptr(phi), ctypes.c_int64(ny), ctypes.c_int64(nx), three, seven, ctypes.byref(opt), ctypes.byref(h)) == 0
    y, x, both = np.ones((ny, nx)), np.ones((ny, nx)), np.ones((2, ny, nx))
    copies()
    lib.amb_get_observable_parts(h, 3, ptr(y), ptr(x))
    apart = copies()
    lib.amb_get_observable(h, 3, ptr(both))
    out.append([apart, copies(), bool((y == 0).all() and (x == 0).all() and (both == 0).all())])
print(json.dumps(out))
""")
    assert out == [[1, 1, True], [1, 1, True], [2, 1, True], [2, 1, True]]
