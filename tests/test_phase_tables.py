"""The engine's host code over a model of the HIP runtime (tests/c/phase_tables.hip):
tables of every route, memory of failed first uses, what streams and events
order.  The model holds a stream's work back until something waits for it, so
an ordering that is missing shows as wrong bytes on the CPU."""
import subprocess
from pathlib import Path

import pytest

from suika_amd.build import INCLUDE, hipcc_path

SRC = Path(__file__).parent / "c" / "phase_tables.hip"


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    out = tmp_path_factory.mktemp("phase_tables")
    for cmd in ([hipcc_path(), "--offload-host-only", "-O2", "-g", "-std=c++17", f"-I{INCLUDE}",
                 f"-I{SRC.parents[2] / 'suika_amd' / 'csrc'}", "-x", "hip", "-c", str(SRC), "-o", str(out / "model.o")],
                # the device code's image, which the host-only object names, is never loaded
                ["g++", "-no-pie", str(out / "model.o"), "-Wl,--unresolved-symbols=ignore-all", "-o", str(out / "model")]):
        res = subprocess.run(cmd, capture_output=True, text=True)
        assert res.returncode == 0, res.stdout + res.stderr
    return out / "model"


@pytest.mark.parametrize("scenario", ["routes", "capture_fails", "two_streams_small", "two_streams_large"])
def test_scenario(model, scenario):
    res = subprocess.run([str(model), scenario], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0 and res.stdout.endswith("ok\n"), res.stdout + res.stderr
