"""Which pass of a transform goes by the direct sum and which by the staged
kernels (fft_direct in kernels.hip), at sizes measured both ways.  The library
runs on the stand-in for the HIP runtime (hip_stub/hip_stub.c), which notes
the kernels launched."""
import json
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# refocus of Nx x Ny at n wavelengths (4 planes each): rows and columns; True: staged.  Times of the row or column pass
# direct / staged in us, or the rates
REFOCUS = [
    ((161, 161), 1, True, True),       # rows of 644 lines, 512 of them 10.8 / 8.6
    ((161, 16), 1, False, True),       # 64 lines 7.9 / 8.2
    ((64, 64), 1, True, True),         # powers of two are always staged
    ((100, 100), 1, True, True),       # and so are lengths of factors up to 13
    ((521, 64), 1, False, True),       # 256 lines 1 / 0.72
    ((521, 64), 4, True, True),        # 1024 lines 1 / 1.65
    ((71, 23), 1, False, True),        # 92 lines 1 / 0.57
    ((71, 64), 16, True, True),        # 4096 lines 1 / 1.77
    ((23, 64), 2, False, True),        # 512 lines 1 / 0.79
    ((1201, 300), 1, False, True),     # a long prime: 1024 lines 1 / 0.83
    ((1201, 300), 16, False, True),    # 16384 lines 9170 / 11600
    ((586, 4), 1, True, True),         # 16 lines 1 / 1.85
    ((2039, 64), 1, False, True),
    ((64, 1361), 1, True, True),       # 256 columns (1301 points) 1 / 1.67
    ((16, 1409), 1, True, False),      # 64 columns 557 / 626
    ((64, 1409), 2, True, True),       # 512 columns 932 / 640
    ((64, 17), 8, True, True),         # 2048 columns 1 / 1.42
    ((4, 23), 256, True, False),       # 4096 columns, four a plane 1 / 0.89
]

DRIVER = """
import ctypes, json, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_name.restype = ctypes.c_char_p
sys.path.insert(0, sys.argv[2])
from nemaktis_amd import viewer

for (nx, ny), nwl, _, _ in json.loads(sys.argv[3]):
    of = viewer.OpticalFields(wavelengths=[0.5 + 0.0001 * k for k in range(nwl)], max_NA_objective=0.6,
                              max_NA_condenser=0.0, N_radial_wavevectors=1, n_out=1.0,
                              mesh_lengths=(0.1 * (nx - 1), 0.1 * (ny - 1)), mesh_dimensions=(nx, ny))
    of.focus_fields(0.5)
    print("route", json.dumps([stub.stub_name(i).decode() for i in range(stub.stub_kernels()) if stub.stub_seen(i)]))
"""


def test_routes(tmp_path):
    if not shutil.which("gcc"):
        pytest.skip("gcc is not available")
    so = str(tmp_path / "libhip_stub.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", so, os.path.join(ROOT, "tests", "hip_stub", "hip_stub.c")],
                   check=True)
    r = subprocess.run([sys.executable, "-c", DRIVER, so, ROOT, json.dumps(REFOCUS)], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    runs = [json.loads(line[6:]) for line in r.stdout.splitlines() if line.startswith("route ")]
    assert len(runs) == len(REFOCUS)
    got = []
    for job, names in zip(REFOCUS, runs):
        rows, cols = (any(k in n for n in names) for k in ("k_fft_rows", "k_view_columns"))
        assert (rows and cols) != any("k_dft_lines" in n for n in names)
        got.append(job[:2] + (rows, cols))
    assert got == REFOCUS
