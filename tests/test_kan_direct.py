"""efficient_kan's direct fp32 path (spline orders 1 to 4, any knot count, small batches):
row blocks, column tiles, feature chunks and basis groups at their edges, against the fp64
oracle at the task tolerance (atol = rtol = 1e-5: the path's fp32 sums of at most a few
hundred terms of size below one round to about 1e-6).  The fast path's ragged tiles are
covered at batches large enough to take it."""
import ctypes
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

from cob_amd import capi, inputs, tasks
from cob_amd.grader.tolerance import tally
from oracle import exact

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parents[1]

# (B, I, O, grid_size, order, knots): 16, 32 and 64 row blocks and one more; 64 columns and
# one on either side; chunks of 4, 8 and 16 features cut short, with C odd so that a run ends
# inside a 16-byte unit; C on both sides of each group of four, up to 31.
SHAPES = [
    (1, 1, 1, 3, 1, "uniform"), (16, 16, 64, 1, 3, "uniform"), (17, 17, 65, 2, 3, "random"),
    (32, 15, 63, 5, 3, "uniform"), (33, 31, 64, 6, 3, "random"), (64, 13, 129, 4, 4, "uniform"),
    (65, 7, 30, 11, 2, "random"), (15, 9, 66, 13, 3, "random"), (16, 33, 70, 14, 3, "uniform"),
    (3, 101, 67, 15, 4, "random"), (31, 45, 80, 17, 4, "uniform"), (130, 21, 64, 22, 2, "random"),
    (5, 50, 33, 29, 1, "uniform"), (40, 18, 90, 25, 3, "uniform"), (70, 6, 17, 29, 1, "random"),
    (9, 1030, 40, 5, 3, "uniform"), (200, 333, 131, 10, 1, "uniform"), (300, 64, 96, 8, 3, "random"),
    (4097, 101, 301, 5, 3, "uniform"), (2050, 70, 1025, 8, 3, "random"),  # the fast path
]


@pytest.mark.parametrize("B,I,O,G,K,knots", SHAPES)
def test_direct_shapes(lib, B, I, O, G, K, knots):
    print(f"\n[kan_direct] B{B} I{I} O{O} G{G} K{K} {knots}", flush=True)
    inp = inputs.make_inputs("efficient_kan", dict(name="d", seed=31 * B + I, B=B, I=I, O=O, grid_size=G,
                                                   spline_order=K, x_range=1.3))
    if knots == "random":
        g = torch.Generator().manual_seed(B)
        step = torch.rand(I, G + 2 * K + 1, generator=g) + 0.25
        inp["grid"] = (torch.cumsum(step, 1) * (3.0 / step.sum(1, keepdim=True)) - 1.5).contiguous()
    inp["x"][0, 0] = inp["grid"][0, K]  # on a knot
    want = exact.efficient_kan(inp)["out"]
    first = None
    for _ in range(2):
        got = capi.run_op(lib, "efficient_kan", inp)["out"].cpu().numpy()
        t = tally(got, want, tasks.load_task("efficient_kan")["tolerance"])
        assert t["mismatched"] == 0, t
        first = got if first is None else first
        assert np.array_equal(got, first)


@pytest.mark.parametrize("B,K", [(8, 3), (70, 2)])
def test_direct_special_inputs(lib, B, K):
    """An infinite or NaN x makes its row NaN and no other; x past fp16's range and weights
    spanning more than 2^24 are ordinary fp32 values."""
    print(f"\n[kan_direct] special inputs B{B} K{K}", flush=True)
    inp = inputs.make_inputs("efficient_kan", dict(name="d", seed=5, B=B, I=40, O=70, grid_size=6, spline_order=K))
    inp["base_weight"][3] *= 2.0 ** -40
    inp["spline_weight"][3, ::2] *= 2.0 ** -40
    inp["x"][4, 5] = 1e5
    want = exact.efficient_kan(inp)["out"]
    bad = {1: float("inf"), 2: float("-inf"), 3: float("nan")}
    for row, v in bad.items():
        inp["x"][row, 11] = v
    got = capi.run_op(lib, "efficient_kan", inp)["out"].cpu().numpy()
    assert np.isnan(got[list(bad)]).all()
    # Row 4 holds 1e5 * Wb, up to 1.6e4: its bound is fp32 roundings of that.
    rel = np.abs(got[4] - want[4]) / np.abs(want[4]).max()
    keep = [r for r in range(B) if r not in bad and r != 4]
    t = tally(got[keep], want[keep], tasks.load_task("efficient_kan")["tolerance"])
    assert t["mismatched"] == 0 and rel.max() < 1e-6, (t, rel.max())


CAPTURE = """
import sys; sys.path.insert(0, {root!r})
import __graft_entry__; __graft_entry__.load_package()
import torch
from cob_amd import capi, inputs
lib = capi.load()
B, I, O, G, K = {shape}
inp = inputs.make_inputs("efficient_kan", dict(name="c", seed=3, B=B, I=I, O=O, grid_size=G, spline_order=K))
args = capi.device_args("efficient_kan", inp)
out = args["out"] = torch.zeros(B, O, device="cuda")
g = torch.cuda.CUDAGraph()
with torch.cuda.graph(g):
    capi.call(lib, "efficient_kan", args)   # the process's first call: no memory to split with
got = []
for _ in range(3):
    out.zero_()
    g.replay()
    torch.cuda.synchronize()
    got.append(out.clone())
capi.call(lib, "efficient_kan", args)       # eager: allocates, splits
torch.cuda.synchronize()
assert all(torch.equal(t, got[0]) for t in got)
assert torch.equal(got[0], out)
g.replay()
torch.cuda.synchronize()
assert torch.equal(out, got[0])
print("captured")
"""


# Other spline orders and finer knots (one, two and four row blocks; few splits and many), and
# small batches of a shape that the packed path also takes.
@pytest.mark.parametrize("shape", [(100, 64, 96, 7, 2), (16, 100, 70, 12, 3), (32, 333, 130, 20, 3), (9, 50, 33, 1, 4),
                                   (8, 256, 256, 5, 3), (130, 96, 100, 8, 3)])
def test_direct_first_call_in_a_capture(lib, shape):
    """A capture may allocate nothing: a tile's one workgroup then takes all splits, in a process
    of its own where no earlier call has grown the memory, and gives the eager call's bits."""
    print(f"\n[kan_direct] first call under capture {shape}", flush=True)
    r = subprocess.run([sys.executable, "-c", CAPTURE.format(root=str(ROOT), shape=shape)], capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0 and "captured" in r.stdout, (r.stdout[-500:], r.stderr[-2000:])


def test_direct_few_splits_after_many(lib):
    """A call split in 2 (or 3) after one split in 16 on the same stream: the sum reads no more
    than its own splits, whatever the earlier call left behind them in the stream's scratch."""
    print("\n[kan_direct] few splits after many", flush=True)
    many = inputs.make_inputs("efficient_kan", dict(name="d", seed=77, B=512, I=80, O=512, grid_size=12, spline_order=3))
    many["base_weight"] = many["base_weight"] * 100.0
    for B, I in [(70, 5), (70, 9), (20, 17), (3, 17)]:
        few = inputs.make_inputs("efficient_kan", dict(name="d", seed=78, B=B, I=I, O=30, grid_size=12, spline_order=3))
        want = exact.efficient_kan(few)["out"]
        capi.run_op(lib, "efficient_kan", many)
        got = capi.run_op(lib, "efficient_kan", few)["out"].cpu().numpy()
        t = tally(got, want, tasks.load_task("efficient_kan")["tolerance"])
        assert t["mismatched"] == 0, (B, I, t)


def test_direct_on_many_streams(lib):
    """Ten streams at once, more than hold scratch memory, in 2 to 16 splits (arrival counters)
    and more (a second launch): every call's result is its own, also when repeated."""
    print("\n[kan_direct] ten streams", flush=True)
    streams = [torch.cuda.Stream() for _ in range(10)]
    args = []
    for k in range(10):
        B, I, O = [(70, 9, 30), (300, 40, 128), (20, 333, 131), (512, 60, 256), (5, 208, 448)][k % 5]
        inp = inputs.make_inputs("efficient_kan", dict(name="d", seed=60 + k, B=B, I=I, O=O, grid_size=12, spline_order=3))
        a = capi.device_args("efficient_kan", inp)
        a["out"] = torch.zeros(B, O, device="cuda")
        args.append((inp, a))
    torch.cuda.synchronize()
    for _ in range(3):
        for s, (_, a) in zip(streams, args):
            capi.call(lib, "efficient_kan", a, s.cuda_stream)
    torch.cuda.synchronize()
    for inp, a in args:
        assert torch.equal(a["out"], capi.run_op(lib, "efficient_kan", inp)["out"])
        t = tally(a["out"].cpu().numpy(), exact.efficient_kan(inp)["out"], tasks.load_task("efficient_kan")["tolerance"])
        assert t["mismatched"] == 0, t


def test_direct_on_streams_that_come_and_go(lib):
    """Twelve streams one after another, each destroyed once its calls have completed, then the
    default one: their scratch regions change hands."""
    print("\n[kan_direct] streams that come and go", flush=True)
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    cases = []
    for B, I, O in [(300, 40, 128), (20, 333, 131)]:
        inp = inputs.make_inputs("efficient_kan", dict(name="d", seed=90 + B, B=B, I=I, O=O, grid_size=12, spline_order=3))
        a = capi.device_args("efficient_kan", inp)
        a["out"] = torch.zeros(B, O, device="cuda")
        cases.append((a, exact.efficient_kan(inp)["out"]))
    torch.cuda.synchronize()
    for k in range(13):
        s = ctypes.c_void_p()
        if k < 12:
            assert hip.hipStreamCreate(ctypes.byref(s)) == 0
        for a, _ in cases:
            a["out"].zero_()
        torch.cuda.synchronize()
        for _ in range(2):
            for a, _ in cases:
                capi.call(lib, "efficient_kan", a, s.value or 0)
        assert hip.hipStreamSynchronize(s) == 0
        if k < 12:
            assert hip.hipStreamDestroy(s) == 0
        for a, want in cases:
            t = tally(a["out"].cpu().numpy(), want, tasks.load_task("efficient_kan")["tolerance"])
            assert t["mismatched"] == 0, (k, t)


def test_small_batch_with_repeated_knots(lib):
    """The packed path leaves out an empty interval's terms; a small batch of its shape, which
    takes the direct path, gives the same values as the packed path's rows."""
    print("\n[kan_direct] repeated knots of a packed shape", flush=True)
    inp = inputs.make_inputs("efficient_kan", dict(name="d", seed=6, B=4096, I=70, O=300, grid_size=5, spline_order=3))
    inp["grid"] = inp["grid"].clone()
    inp["grid"][:, :4] = inp["grid"][:, 3:4]    # clamped ends
    inp["grid"][:, -4:] = inp["grid"][:, -4:-3]
    packed = capi.run_op(lib, "efficient_kan", inp)["out"].cpu().numpy()
    few = dict(inp, x=inp["x"][:9].contiguous(), B=9)
    got = capi.run_op(lib, "efficient_kan", few)["out"].cpu().numpy()
    t = tally(got, packed[:9].astype(np.float64), tasks.load_task("efficient_kan")["tolerance"])
    assert t["mismatched"] == 0 and np.isfinite(got).all(), t
