"""reward_to_go on rows at any alignment and on few long rows split over workgroups: part and
chunk edges, odd row lengths, offset pointers, streams and captures, against the fp64 oracle
at the task tolerance (atol = rtol = 1e-5; the fp32 steps from fp64 carries measure at most
0.25 of it at these discounts)."""
import ctypes

import numpy as np
import pytest
import torch

from cob_amd import capi, inputs, tasks
from cob_amd.grader.tolerance import tally
from oracle import exact

pytestmark = pytest.mark.gpu
TOL = tasks.load_task("reward_to_go")["tolerance"]


def _case(B, T, gamma=0.99, done_p=0.001, seed=0):
    return inputs.make_inputs("reward_to_go", dict(name="r", seed=seed + B + T, B=B, T=T, gamma=gamma, done_p=done_p))


# Whole rows at odd lengths (every launch shape); the split from 12289 steps on, parts of 4 and
# of 16 chunks, last parts of one chunk, of one step and whole; more than 64 parts in a row.
SHAPES = [(3, 255), (2, 257), (5, 511), (3, 1023), (4, 2047), (9, 4097), (300, 1999), (6, 12288), (6, 12289),
          (1, 12545), (2, 13312), (3, 13313), (1, 65537), (2, 70001), (1, 131072), (40, 28672), (40, 28673),
          (33, 32769), (256, 12290), (257, 12290)]


@pytest.mark.parametrize("B,T", SHAPES)
def test_rows(lib, B, T):
    print(f"\n[rtg] B{B} T{T}", flush=True)
    inp = _case(B, T)
    want = exact.reward_to_go(inp)["output"]
    outs = [capi.run_op(lib, "reward_to_go", inp)["output"].cpu().numpy() for _ in range(2)]
    assert np.array_equal(*outs)
    t = tally(outs[0], want, TOL)
    assert t["mismatched"] == 0 and t["worst"] < 0.25, t


@pytest.mark.parametrize("gamma,done_p", [(1.0, 0.01), (0.0, 0.1), (-0.9, 0.01), (1.25, 0.2), (0.999, 0.0)])
def test_split_discounts(lib, gamma, done_p):
    """Discounts above 1 in size (whole rows only), zero, negative and slow ones."""
    print(f"\n[rtg] gamma {gamma} done {done_p}", flush=True)
    inp = _case(2, 20001, gamma, done_p)
    t = tally(capi.run_op(lib, "reward_to_go", inp)["output"].cpu(), exact.reward_to_go(inp)["output"], TOL)
    assert t["mismatched"] == 0, t


@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("B,T", [(3, 4096), (2, 16384)])
def test_offset_pointers(lib, B, T, off):
    print(f"\n[rtg] B{B} T{T} offset {off}", flush=True)
    inp = _case(B, T)
    n = B * T
    r = torch.zeros(n + 8, device="cuda")
    d = torch.zeros(n + 8, dtype=torch.bool, device="cuda")
    out = torch.full((n + 8,), 7.0, device="cuda")
    r[off:off + n] = inp["reward"].flatten().cuda()
    d[off:off + n] = inp["done"].flatten().cuda()
    capi.call(lib, "reward_to_go", dict(reward=r[off:], done=d[off:], gamma=inp["gamma"], B=B, T=T, output=out[off:]))
    torch.cuda.synchronize()
    t = tally(out[off:off + n].reshape(B, T).cpu(), exact.reward_to_go(inp)["output"], TOL)
    assert t["mismatched"] == 0, t
    assert bool((out[:off] == 7.0).all()) and bool((out[off + n:] == 7.0).all())


def test_split_on_many_streams(lib):
    """Ten streams at once, more than hold scratch memory: every call's result is its own."""
    print("\n[rtg] ten streams", flush=True)
    streams = [torch.cuda.Stream() for _ in range(10)]
    args = []
    for k in range(10):
        inp = _case(4, 40_000 + 4 * k, seed=k)
        a = capi.device_args("reward_to_go", inp)
        a["output"] = torch.zeros(4, inp["T"], device="cuda")
        args.append((inp, a))
    torch.cuda.synchronize()
    for _ in range(3):
        for s, (_, a) in zip(streams, args):
            capi.call(lib, "reward_to_go", a, s.cuda_stream)
    torch.cuda.synchronize()
    for inp, a in args:
        t = tally(a["output"].cpu(), exact.reward_to_go(inp)["output"], TOL)
        assert t["mismatched"] == 0, t


def test_split_on_streams_that_come_and_go(lib):
    """Twelve streams one after another, each destroyed once its call has completed."""
    print("\n[rtg] streams that come and go", flush=True)
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    inp = _case(4, 50_000)
    a = capi.device_args("reward_to_go", inp)
    out = a["output"] = torch.zeros(4, 50_000, device="cuda")
    torch.cuda.synchronize()
    want = exact.reward_to_go(inp)["output"]
    for _ in range(12):
        s = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(s)) == 0
        out.zero_()
        torch.cuda.synchronize()
        for _ in range(2):
            capi.call(lib, "reward_to_go", a, s.value)
        assert hip.hipStreamSynchronize(s) == 0
        assert hip.hipStreamDestroy(s) == 0
        assert tally(out.cpu(), want, TOL)["mismatched"] == 0


def test_split_under_capture(lib):
    """A captured call takes the whole-row form, which holds no scratch memory, and replays."""
    print("\n[rtg] capture", flush=True)
    inp = _case(3, 30_000)
    a = capi.device_args("reward_to_go", inp)
    out = a["output"] = torch.zeros(3, 30_000, device="cuda")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        capi.call(lib, "reward_to_go", a)
    for k in range(3):
        new = _case(3, 30_000, seed=50 + k)
        a["reward"].copy_(new["reward"])
        a["done"].copy_(new["done"])
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        t = tally(out.cpu(), exact.reward_to_go(new)["output"], TOL)
        assert t["mismatched"] == 0, t
