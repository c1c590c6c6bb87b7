"""The rules of csrc/route.h, compiled for the host, at sizes where both sides were timed on the device:
the rule takes the faster one.
"""
import ctypes
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "e2e-browser-voice-agent_amd" / "csrc"

SHIM = """
#include "route.h"
extern "C" {
int mv(int N, int nb) { return q4::mv_quantizes_itself(N, nb); }
}
"""


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    d = tmp_path_factory.mktemp("route")
    (d / "shim.cpp").write_text(SHIM)
    so = d / "shim.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", str(CSRC), "-o", str(so),
                    str(d / "shim.cpp")], check=True)
    return ctypes.CDLL(str(so))


# rows, blocks per row, microseconds with a quantize launch of its own, quantized by each workgroup
MATVEC = [(128, 1, 5.52, 3.59), (896, 28, 6.00, 4.34), (151936, 4, 7.28, 5.92), (151936, 28, 15.64, 13.90),
          (151936, 48, 25.47, 23.98), (151936, 63, 33.23, 32.06), (896, 64, 5.91, 3.99), (896, 152, 8.70, 6.18),
          (17920, 64, 12.76, 12.19), (28672, 64, 16.97, 16.72), (65536, 64, 32.88, 35.31), (151936, 64, 68.96, 80.53),
          (28672, 100, 24.19, 23.08), (65536, 100, 46.06, 48.62), (28672, 152, 32.71, 31.78), (80000, 152, 76.51, 79.88),
          (1536, 280, 13.1, 9.9), (20480, 280, 53.39, 52.00), (40960, 280, 97.52, 100.45), (151936, 280, 353.98, 373.20),
          (16384, 400, 59.00, 57.32), (40960, 400, 137.59, 140.23), (12288, 480, 54.20, 51.96),
          (24576, 480, 99.69, 101.22), (80000, 480, 314.01, 331.95)]


@pytest.mark.parametrize("rows,blocks,launch,itself", MATVEC)
def test_matvec_quantize(route, rows, blocks, launch, itself):
    assert bool(route.mv(rows, blocks)) == (itself < launch)


def test_matvec_quantize_limits(route):
    assert not route.mv(1, 481)
    assert route.mv(14656, 480) and not route.mv(14657, 480)
