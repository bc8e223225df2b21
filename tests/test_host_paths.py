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


@pytest.mark.parametrize("op,args", [("efficient_kan", FINE_KNOTS), ("efficient_kan", SMALL_BATCH)])
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


@pytest.mark.parametrize("capturing", [0, 1])
def test_split_rows_use_no_memory_of_the_library(host, capturing):
    """Few long rows take two launches on any stream, under capture too, and allocate nothing;
    an output that shares memory with an input takes the whole-row form."""
    out = host([put("capturing", 4, capturing)] + [call("reward_to_go", stream=s, **FEW_LONG_ROWS) for s in (4, 0, 2)]
               + [call("reward_to_go", stream=4, reward=1 << 41, output=(1 << 41) + 64, **FEW_LONG_ROWS),
                  call("reward_to_go", stream=4, done=(1 << 41) + 4 * 16 * 65536 - 4, output=1 << 41, **FEW_LONG_ROWS),
                  call("reward_to_go", stream=4, done=(1 << 41) + 4 * 16 * 65536, output=1 << 41, **FEW_LONG_ROWS)])
    assert [len(kernels(s)) for s in out[1:]] == [2, 2, 2, 1, 1, 2]
    assert not any(line.startswith("malloc") for s in out for line in s["log"])


def fp8_kernel(host, *sizes, x=0):
    steps = [call("fp8_linear", M=M, K=K, N=N, scale_x=1.0, scale_w=1.0, x_fp8=(1 << 40) + x) for M, K, N in sizes]
    out = host(steps)
    assert all(s["rc"] == 0 for s in out)
    names = [kernels(s) for s in out]
    assert all(len(n) == 1 for n in names)
    return [n[0] for n in names]


# Sides of fp8_linear's rule for at most 64 rows: the skinny kernel where its workgroups fit the
# CUs once (it was up to 25% faster there than the tiles), the tiles beyond.
FP8_SKINNY = [(33, 2048, 64), (33, 4096, 64), (40, 2048, 4096), (40, 1536, 1024), (33, 1024, 512), (48, 2048, 2048), (64, 1024, 512), (64, 2048, 1024),
              (64, 4096, 4096), (64, 8192, 512), (64, 7168, 4096), (56, 704, 1600), (63, 3136, 576), (16, 16384, 4096),
              (32, 8192, 4096), (16, 16384, 8192), (8, 4096, 6144), (48, 8192, 520), (33, 4096, 448), (39, 5536, 1568),
              (16, 4088, 8200), (33, 1016, 4104), (33, 2040, 8000), (48, 4088, 4096), (64, 4088, 1024)]
FP8_TILES = [(40, 1024, 4096), (33, 256, 64), (48, 640, 512), (48, 1280, 1024), (33, 4096, 1024), (48, 2064, 512), (48, 8192, 64), (64, 7168, 504), (33, 256, 4112), (64, 256, 4112), (64, 8192, 5120), (17, 256, 5120),
             (32, 16384, 5120), (1, 256, 7168), (16, 8192, 8192), (16, 16384, 16384), (33, 4088, 4104), (48, 1016, 8200),
             (64, 1016, 4104), (1, 333, 300), (64, 4095, 64), (16, 63, 4096)]


def test_fp8_small_m_routes(host):
    for size, name in zip(FP8_SKINNY, fp8_kernel(host, *FP8_SKINNY)):
        assert "fp8_gemm_skinny" in name, (size, name)
    for size, name in zip(FP8_TILES, fp8_kernel(host, *FP8_TILES)):
        assert "fp8_gemm_mid" in name, (size, name)


def kan_kernel(host, *shapes, order=3):
    """"direct", "fast" (kan_fused) or "rowwise" for (B, I, O, G[, order]) on a fresh library."""
    steps = [call("efficient_kan", B=s[0], I=s[1], O=s[2], grid_size=s[3], spline_order=s[4] if len(s) > 4 else order)
             for s in shapes]
    out = host(steps)
    assert all(s["rc"] == 0 for s in out)
    known = {"kan_directI": "direct", "kan_fused": "fast", "kan_rowwise": "rowwise"}
    return [next(v for k, v in known.items() if any(k in n for n in kernels(s))) for s in out]


# Both sides of efficient_kan's choice between the direct and the fast path, at shapes where one
# of them was measured at least 10% faster.
KAN_DIRECT = [(8, 1024, 1024, 5), (128, 1024, 1024, 5), (256, 256, 512, 8), (6889, 128, 64, 5), (4096, 512, 64, 3),
              (341, 65, 1606, 5), (1024, 1024, 1024, 16), (16, 8, 8, 5), (1852, 64, 512, 8, 2)]
KAN_FAST = [(1710, 1000, 100, 5), (1499, 1000, 100, 5), (6561, 32, 128, 5), (2823, 32, 320, 3), (2114, 256, 256, 3),
            (716, 1856, 192, 5), (512, 1024, 1024, 5), (4096, 256, 512, 8), (8192, 1024, 1024, 5)]


def test_kan_routes(host):
    assert kan_kernel(host, *KAN_DIRECT) == ["direct"] * len(KAN_DIRECT)
    assert kan_kernel(host, *KAN_FAST) == ["fast"] * len(KAN_FAST)


def fine(stream):
    return call("efficient_kan", stream=stream, **FINE_KNOTS)


def split(step):
    """Whether a FINE_KNOTS call ran with its features split over workgroups (128 tiles)."""
    assert step["rc"] == 0
    line, = [line for line in step["log"] if "kan_directI" in line]
    return int(line.split("grid ")[1].split()[0]) > 128


def test_one_streams_calls_carry_no_event(host):
    out = host([fine(3), fine(3)])
    assert all(split(s) and not any(line.endswith("event") for line in s["log"]) for s in out)


def test_streams_give_their_scratch_back(host):
    """Twelve streams, each done when the next one calls: all of them split, on eight regions.
    The first one's only use had no event, so its region stays its own."""
    out = host([fine(s) for s in range(3, 15)] + [fine(3)])
    assert all(split(s) for s in out)
    assert sum(line.startswith("malloc") for s in out for line in s["log"]) <= 16  # regions and one growth each
    assert not any(line.startswith("malloc") for s in out[8:] for line in s["log"])
    assert all(s["log"][-1].endswith("event") for s in out[1:])


def test_busy_streams_keep_their_scratch(host):
    """No region is taken from a stream whose last call has not completed, and asking about
    them leaves another stream's capture whole; the owners still have theirs afterwards."""
    busy = [put("busy", s, 1) for s in range(3, 11)] + [put("capturing", 30, 1), put("global_capture", 1)]
    out = host([fine(s) for s in range(3, 11)] + busy + [fine(20), fine(5)])
    assert not split(out[-2]) and split(out[-1])
    assert not any(line.startswith("capture_broken") for line in out[-2]["log"]), out[-2]["log"]


def test_the_least_recently_used_scratch_goes_first(host):
    order = [3, 4, 5, 6, 7, 8, 9, 10, 3, 4]  # 5 is the oldest use
    steps = [fine(s) for s in order] + [put("busy", s, 1) for s in range(3, 11) if s not in (5, 9)]
    out = host(steps + [fine(20), fine(9), put("busy", 9, 1), put("busy", 20, 1), fine(5)])
    assert split(out[-5]) and split(out[-4]) and not split(out[-1])


def test_fp8_more_tiles_than_one_launch_takes(host):
    """8.75 M tiles of 128 x 128 by 512 threads (an output of 280 GB): launches of at most 2^32 - 1
    work-items, together all of the tiles."""
    out = host([call("fp8_linear", M=70_000_000, K=1, N=2000, scale_x=1.0, scale_w=1.0)])[0]
    grids = [int(line.split("grid ")[1].split()[0]) for line in out["log"] if line.startswith("launch")]
    assert out["rc"] == 0 and max(grids) * 512 < 2 ** 32 and sum(grids) == 546_875 * 16, out


def test_gpu_tests_reach_the_paths_they_name(host):
    """The shape lists of the GPU tests, by path: a change of the rules shows here."""
    import test_gpu_parity as parity
    import test_gpu_random_cases as rand
    import test_gpu_special as special
    import test_graphs as graphs

    def kan(cases):
        return set(kan_kernel(host, *[tuple(c) for c in cases]))

    def sizes(case):
        return [case[k] for k in ("B", "I", "O")] + [case.get("grid_size", 5), case.get("spline_order", 3)]

    assert kan(s[:5] for s in parity.KAN_SHAPES) == {"direct"}
    assert kan(s[:5] for s in parity.KAN_PACKED_SHAPES) == {"fast"}
    assert kan(s[:5] for s in parity.KAN_ROWWISE_SHAPES) == {"rowwise"}
    assert kan_kernel(host, *[(B, 1024, 1024, 5) for B in parity.JITTER_ROWS]) == ["direct", "fast"]
    assert kan(sizes(c) for _, c in rand.PACKED_CASES) == {"fast"}
    assert kan([sizes(graphs.SMALL["efficient_kan"])]) == {"direct"} and kan([sizes(graphs.LARGE["efficient_kan"])]) == {"fast"}
    assert kan_kernel(host, *special.KAN_PATHS.values()) == list(special.KAN_PATHS)

    def fp8(*cases):
        names = ["fp8_gemm_skinny_flat", "fp8_gemm_skinny", "fp8_gemm_mid", "fp8_gemm_half", "fp8_gemm_wide"]
        return [next(n for n in names if n in k)[9:] for k in fp8_kernel(host, *[c[:3] for c in cases])]

    assert fp8(*special.FP8_KERNELS.values()) == ["skinny_flat", "mid", "mid", "half", "wide"]
    assert set(fp8(*parity.FP8_SHAPES)) == {"skinny_flat", "skinny", "mid", "half", "wide"}
    three = [c for c in parity.FP8_SHAPES if c[:3] in ((40, 2064, 64), (33, 1312, 20))]
    assert len(three) == 2 and all("skinny_flatILi3E" in k for k in fp8_kernel(host, *[c[:3] for c in three]))
    assert fp8((70, 0, 72), (2200, 0, 4000), (2000, 0, 4000), (16, 0, 40)) == ["mid", "wide", "half", "skinny_flat"]
    large = graphs.LARGE["fp8_linear"]
    assert fp8((large["M"], large["K"], large["N"])) == ["wide"]
