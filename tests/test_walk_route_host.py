"""Which line solvers an FP64 march at the built-in shapes takes: the walking
ones where they were measured to be the faster (walk_pays in engine.cpp), the
ones on stored stencils elsewhere.  The library runs on the stand-in for the
HIP runtime (hip_stub/hip_stub.c), which notes the kernels launched."""
import json
import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# mesh, directions a wavelength, wavelengths, precision; True: walks.  Times a slab in us, stored / walking
ROUTES = [
    ((65, 65), 1, 1, 64, True),        # 68 / 54
    ((512, 512), 1, 1, 64, True),      # 252 / 173
    ((512, 512), 1, 1, 32, False),     # FP32 keeps the stored stencils
    ((128, 128), 7, 1, 64, True),      # one round of blocks: 120 / 109
    ((192, 26), 7, 1, 64, True),       # 75.6 / 75.7
    ((506, 18), 1, 1, 64, False),      # 73.1 / 74.8
    ((1000, 17), 1, 1, 64, False),     # 94.5 / 96.1
    ((1001, 49), 1, 1, 64, False),     # 115.8 / 117
    ((339, 19), 1, 1, 64, False),      # 68 / 64, left out with the strips
    ((351, 25), 1, 1, 64, True),       # 68.1 / 64.7
    ((18, 506), 1, 1, 64, True),
    ((401, 66), 1, 7, 64, True),       # 178 / 149
    ((1001, 41), 1, 3, 64, False),     # 145 / 159
    ((601, 21), 1, 7, 64, False),      # 121 / 139
    ((13, 1001), 1, 7, 64, True),      # 232 / 163
    ((1001, 13), 1, 7, 64, False),     # 124 / 163
    ((601, 131), 7, 1, 64, True),      # 505 / 479
    ((1001, 201), 7, 1, 64, True),     # 1085 / 1075
    ((128, 128), 7, 21, 64, True),     # 1411 / 1215
    ((1001, 121), 7, 3, 64, False),    # 1715 / 1797
    ((1001, 171), 7, 3, 64, False),    # 2730 / 2780
    ((1001, 301), 7, 3, 64, True),     # 5230 / 5060
    ((601, 65), 7, 1, 64, False),      # 225 / 256
    ((301, 41), 7, 1, 64, False),      # 113 / 125
    ((1000, 12), 37, 1, 64, False),    # 271 / 583
    ((201, 201), 37, 1, 64, True),     # 981 / 940
    ((301, 601), 19, 1, 64, True),     # 2540 / 2320
    ((341, 601), 61, 1, 64, False),    # 12380 / 13020
    ((385, 301), 61, 1, 64, True),     # 5500 / 5170
    ((1001, 301), 37, 1, 64, False),   # 9020 / 10930
    ((257, 1001), 37, 1, 64, False),   # 8210 / 8520
    ((65, 1001), 37, 1, 64, False),    # 1870 / 2060
    ((1026, 65), 1, 1, 64, False),     # no shape above 1024 points
    ((8, 65), 1, 1, 64, False),        # nor below 8
    ((9, 65), 1, 1, 64, True),
    ((3, 65), 1, 1, 64, False),        # an axis that is not periodic
]

# mesh, directions, wavelengths: whether FP32 takes the register-lean solvers.  Fuller / lean, us a slab or rates
LEAN = [
    ((257, 257), 1, 1, True),          # 109 / 106
    ((257, 101), 1, 1, True),
    ((334, 52), 1, 1, False),          # 69.0 / 71.5
    ((401, 401), 1, 1, False),         # 1 / 0.99
    ((200, 401), 1, 1, True),          # 1 / 1.07
    ((512, 512), 1, 1, False),         # 188 / 191
    ((401, 102), 1, 2, False),         # 1 / 0.99
    ((401, 161), 1, 2, True),          # 1 / 1.15
    ((301, 203), 7, 3, True),          # 631 / 554
    ((513, 513), 7, 1, True),
    ((514, 514), 7, 1, False),
]

DRIVER = """
import ctypes, json, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_name.restype = ctypes.c_char_p
sys.path.insert(0, sys.argv[2])
import numpy as np
from nemaktis_amd import _lib, bpm_backend, fields

_lib.load()
print("holds", json.dumps([stub.stub_name(i).decode() for i in range(stub.stub_kernels())]))
for (nx, ny), nq, nwl, precision, _ in json.loads(sys.argv[3]):
    dims = (nx, ny, 2)
    s = fields.make_settings(dims, (0.1, 0.1, 0.1), [0.5 + 0.01 * k for k in range(nwl)],
                             wavevectors=[(0.01 * k, 0.0) for k in range(nq)])
    lc = np.zeros((2 * nx * ny, 3))
    with bpm_backend.Context(json.dumps(s), lc, int(np.prod(fields.output_shape(s))), precision=precision,
                             wl_batch=0) as c:
        c.propagate()
    names = {stub.stub_name(i).decode(): stub.stub_blocks(i) for i in range(stub.stub_kernels()) if stub.stub_seen(i)}
    print("route", json.dumps(names))
"""


def launched(so, jobs):
    """The mangled names of the library's kernels, and of those that each job launches with the blocks of the last
    launch."""
    r = subprocess.run([sys.executable, "-c", DRIVER, so, ROOT, json.dumps(jobs)], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    lines = [line.split(" ", 1) for line in r.stdout.splitlines()]
    return json.loads(lines[0][1]), [json.loads(v) for k, v in lines if k == "route"]


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    if not shutil.which("gcc"):
        pytest.skip("gcc is not available")
    so = str(tmp_path_factory.mktemp("stub") / "libhip_stub.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", so, os.path.join(ROOT, "tests", "hip_stub", "hip_stub.c")],
                   check=True)
    return so


def test_routes(stub):
    got = []
    for job, names in zip(ROUTES, launched(stub, ROUTES)[1]):
        walks = any("k_walk" in n for n in names)
        stored = any("k_xsolve" in n or "k_ysolve" in n for n in names)
        assert walks != stored, (job, names)
        got.append(job[:4] + (walks,))
    assert got == ROUTES


def test_lean_shapes(stub):
    got = []
    for job, names in zip(LEAN, launched(stub, [j[:3] + (32, True) for j in LEAN])[1]):
        lean = {re.search(r"k_ysolveIfLi\d+ELi[01]ELi([01])E", n).group(1) for n in names if "k_ysolve" in n}
        assert len(lean) == 1
        got.append(job[:3] + (lean == {"1"},))
    assert got == LEAN


def test_short_lines_keep_whole_strips(stub):
    """FP32, a lone pair: strips of lines under 32 points are not halved (222 x 29 55.3 us a slab, halved 57.3)."""
    short, long = ([b for n, b in names.items() if "k_ysolve" in n][0]
                   for names in launched(stub, [((222, ny), 1, 1, 32, True) for ny in (29, 33)])[1])
    assert 2 * short <= long + 8


def test_the_library_holds_no_walking_kernel_that_nothing_reaches(stub):
    holds = launched(stub, [])[0]
    # FP64 only: the slab material and the kernels of a state with x slow
    x_slow = r"k_(init_fields|pack_fields|boundary|boundary_point|output|bulk_plane)I%sLb1E"
    assert not [n for n in holds if re.search("k_slab_materialIf|" + x_slow % "f", n)]
    assert len([n for n in holds if re.search("k_slab_materialId|" + x_slow % "d", n)]) == 7
    # two lines a block have chunks of more than 3 points
    assert not [n for n in holds if re.search(r"k_walkILi[23]ELi2E", n)]


def test_gpu_tests_cover_every_instance(stub):
    """k_walk's instances in the jobs of test_gpu_walk.test_every_kernel_instance."""
    from test_gpu_walk import SHAPES

    holds, runs = launched(stub, [((nx, ny), nq, nwl, 64, True) for nx, ny, nq, nwl in SHAPES])
    instance = re.compile(r"k_walkILi\d+ELi\d+ELi[01]E")
    found = set()
    for (nx, ny, nq, nwl), names in zip(SHAPES, runs):
        got = {m.group() for m in map(instance.search, names) if m}
        assert got, "%d x %d does not walk" % (nx, ny)
        found |= got
    assert found == {m.group() for m in map(instance.search, holds) if m}


def test_bench_names_the_kernels_of_its_512_job(stub):
    sys.path.insert(0, ROOT)
    import bench

    for precision in (64, 32):
        names = " ".join(launched(stub, [((512, 512), 1, 1, precision, True)])[1][0])
        named = bench.KERNELS_WALK if bench.walks(precision, None) else bench.KERNELS
        assert all(named[fam] in names for fam in ("solve_x", "solve_y", "boundary", "coefs"))
