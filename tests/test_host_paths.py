"""The library's host side on the CPU, against a stub HIP runtime (hip_stub.c) that records
launches, allocations and events and answers as one MI355X would."""
import json
import subprocess
import sys
from pathlib import Path

import pytest

from cob_amd import capi

HERE = Path(__file__).resolve().parent
LIB = HERE.parent / "cuda-optimization-benchmark_amd" / "lib" / "libtaskops.so"


@pytest.fixture(scope="session")
def host(tmp_path_factory):
    """Runs steps in a fresh process under the stub and returns their records."""
    stub = tmp_path_factory.mktemp("stub") / "hip_stub.so"
    subprocess.run(["gcc", "-O1", "-std=gnu11", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(HERE / "hip_stub.c"), "-o", str(stub)], check=True)

    def run(steps):
        r = subprocess.run([sys.executable, str(HERE / "host_probe.py"), str(stub), str(LIB)], input=json.dumps(steps),
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-2000:]
        return json.loads(r.stdout)
    return run


CODES = {capi._P: "p", capi._I32: "i", capi._I64: "l", capi._F32: "f"}


def call(op, stream=0, **args):
    """A step: `op` with the given scalars; pointers default to 16-byte aligned addresses that
    nothing reads."""
    sym, params = capi.ENTRY[op]
    vals, base = [], 1 << 40
    for name, t in params:
        base += 1 << 34
        vals.append(args.pop(name, base if t is capi._P else None))
    assert not args and None not in vals, (op, args, vals)
    return {"call": sym, "types": "".join(CODES[t] for _, t in params) + "p", "args": vals + [stream]}


def put(name, *args):
    return {"set": name, "args": list(args)}


def kernels(step):
    return [line.split()[1] for line in step["log"] if line.startswith("launch ")]


FEW_LONG_ROWS = dict(gamma=0.99, B=16, T=65536)
FINE_KNOTS = dict(grid_size=16, spline_order=3, B=1024, I=256, O=512)
SMALL_BATCH = dict(grid_size=5, spline_order=3, B=8, I=1024, O=1024)


@pytest.mark.parametrize("op,args", [("reward_to_go", FEW_LONG_ROWS), ("efficient_kan", FINE_KNOTS),
                                     ("efficient_kan", SMALL_BATCH)])
def test_allocating_leaves_another_streams_capture_alone(host, op, args):
    """A first call on stream 3 allocates while stream 4 captures (the stub, like the runtime,
    breaks the capture for an allocation in the default capture mode)."""
    out = host([put("capturing", 4, 1), put("global_capture", 1), call(op, stream=3, **args)])[-1]
    assert out["rc"] == 0
    assert any(line.startswith("malloc") for line in out["log"])
    assert not any(line.startswith("capture_broken") for line in out["log"]), out["log"]


@pytest.mark.parametrize("op,args", [("reward_to_go", FEW_LONG_ROWS), ("efficient_kan", FINE_KNOTS),
                                     ("efficient_kan", SMALL_BATCH)])
def test_a_capturing_stream_allocates_nothing(host, op, args):
    out = host([put("capturing", 4, 1), put("global_capture", 1), call(op, stream=4, **args)])[-1]
    assert out["rc"] == 0 and not any(line.startswith(("malloc", "capture_broken")) for line in out["log"]), out["log"]
