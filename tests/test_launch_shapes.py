"""The launches of a call, recorded on the host (tests/cpp/launch_recorder.cpp in the place of the HIP runtime): which
kernels a problem takes, and that HIP accepts every grid: not empty, fewer than 2^32 threads along x. No kernel
runs, so the problems may be as large as the entry points take."""
import json
import os
import subprocess
import sys

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))
RECORDER = os.path.join(TESTS, "cpp", "launch_recorder.cpp")
F32, F64, F16, BF16 = range(4)
SUCCESS, INVALID_ARGUMENT = 0, 1

# (a process without torch, whose libraries bring the HIP runtime's own symbols)
CHILD = """
import json, sys
sys.path.insert(0, sys.argv[1])
from launch_child import record
print(json.dumps(record(sys.argv[2], sys.argv[3], json.load(sys.stdin))))
"""


def problem(dim, batch, cin, cout, size, kernel, **kw):
    p = dict(dim=dim, batch=batch, cin=cin, cout=cout, size=size, kernel=kernel, transposed=False, dtype=F32, groups=1,
             og=1, mg=1, flags=0, stride=1, padding=0, dilation=1, out_pad=0, bias=True)
    p.update(kw)
    return p


@pytest.fixture(scope="module")
def record(tmp_path_factory):
    """record(problem) -> {"forward" / "backward": {"status", "error", "launches": [(kernel, grid, block)]}}"""
    import tvdcn
    lib = str(tmp_path_factory.mktemp("recorder") / "launch_recorder.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", RECORDER, "-o", lib], check=True)

    def go(p):
        child = subprocess.run([sys.executable, "-c", CHILD, TESTS, lib, tvdcn.extension.HIP_LIB_PATH],
                               input=json.dumps([p]), stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True,
                               timeout=120)
        assert child.returncode == 0, (child.returncode, child.stderr[-2000:])
        return json.loads(child.stdout)[0]

    return go


@pytest.mark.parametrize("batch", [0, 2])
@pytest.mark.parametrize("cin,dtype", [(8, F32), (8, F16), (64, F32), (64, F64)])
def test_transposed_layer_of_an_empty_input_is_refused(record, cin, dtype, batch):
    """A 4 x 4 kernel gives an empty input an output of 1 x 5 pixels but no column to compute it from: an error, before
    any launch, forward and backward."""
    r = record(problem(2, batch, cin, 4, [0, 4], [4, 4], transposed=True, padding=1, dtype=dtype))
    for call in r.values():
        assert call["status"] == INVALID_ARGUMENT and "positive" in call["error"] and not call["launches"]
