"""A change of launch shapes whose buffers do not fit: the context keeps its
shapes and buffers (include/nemaktis_bpm.h), or, where another user of the
device has taken even those, refuses to march until a change succeeds.  The
library runs on a stand-in for the HIP runtime (hip_stub/hip_stub.c) whose
allocations fail on request; no kernel runs.  In a process of its own, which
loads the stand-in before the library."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = """
import ctypes, json, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_live.restype = ctypes.c_size_t
sys.path.insert(0, sys.argv[2])
import numpy as np
from nemaktis_amd import bpm_backend, fields

to_walk, use_graph = sys.argv[3] == "built-in", sys.argv[4] == "graph"
skip, fail = int(sys.argv[5]), int(sys.argv[6])
dims = (40, 36, 6)
s = fields.make_settings(dims, (0.1, 0.1, 0.1), [0.6], wavevectors=((0.0, 0.0), (0.1, 0.05)))
lc = np.tile([1.0, 0.0, 0.0], (dims[2] * dims[1] * dims[0], 1))
explicit = {"x_chunks": 16, "x_rows": 2, "y_chunks": 16, "y_cols": 8}
first, second = (explicit, None) if to_walk else (None, explicit)

def context(tuning):
    return bpm_backend.Context(json.dumps(s), lc, int(np.prod(fields.output_shape(s))), precision=64,
                               use_graph=use_graph, tuning=tuning)

def marches(c):
    before = stub.stub_launches()
    bytes_ = c.propagate()["footprint_bytes"]
    assert stub.stub_launches() > before or use_graph
    return bytes_

with context(second) as c:
    want = marches(c)
with context(first) as c:
    held, own = stub.stub_live(), marches(c)
    stub.stub_fail(skip, fail)
    try:
        c.set_tuning(second)
        refused = False
    except bpm_backend.BpmBackendError as e:
        refused = True
        assert "out of memory" in str(e), e
    stub.stub_fail(0, 0)
    lost = False
    if refused:
        before = stub.stub_launches()
        try:
            assert marches(c) == own and stub.stub_live() == held
        except bpm_backend.BpmBackendError as e:
            lost = True
            assert stub.stub_launches() == before, "launched without buffers"
        c.set_tuning(second)
    assert marches(c) == want
    c.set_tuning(first)
    assert marches(c) == own and stub.stub_live() == held
assert stub.stub_live() == 0 and stub.stub_unfit() == 0
print("refused" if refused else "switched", "lost" if lost else "kept")
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    if not shutil.which("gcc"):
        pytest.skip("gcc is not available")
    so = str(tmp_path_factory.mktemp("stub") / "libhip_stub.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", so, os.path.join(ROOT, "tests", "hip_stub", "hip_stub.c")],
                   check=True)
    return so


# a change takes two buffers, beside the old ones first (the first failure), then in their place (the second); the third
# failure meets the return to the old ones
@pytest.mark.parametrize("mode", ["eager", "graph"])
@pytest.mark.parametrize("to", ["built-in", "explicit"])
@pytest.mark.parametrize("skip,fail,outcome", [(0, 0, "switched kept"), (0, 1, "switched kept"), (1, 1, "switched kept"),
                                               (0, 2, "refused kept"), (1, 2, "refused kept"), (0, 3, "refused lost"),
                                               (1, 3, "refused lost"), (0, 4, "refused lost")])
def test_failed_allocations(stub, to, mode, skip, fail, outcome):
    r = subprocess.run([sys.executable, "-c", DRIVER, stub, ROOT, to, mode, str(skip), str(fail)],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
    assert r.stdout.strip().endswith(outcome), r.stdout[-3000:]
