"""quantize_e4m3 past one chunk per resident workgroup: the held chunks (registers and LDS), the
chunks read twice, the part chunk, the bounded wait's fallback, a captured graph, and the two
launches beyond, codes and scale equal to torch's cast bit for bit."""
import ctypes

import pytest
import torch

from cob_amd import capi

pytestmark = pytest.mark.gpu
CHUNK = 16384


def _want(x):
    s = torch.tensor(448.0 / max(x.abs().max().item(), 1e-9), dtype=torch.float32, device="cuda")
    return (x * s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8), s


def _run(lib, x, n):
    q = torch.full((n + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    s = torch.zeros(1, device="cuda")
    capi.call(lib, "quantize_e4m3", dict(x=x, n=n, q=q, scale=s))
    torch.cuda.synchronize()
    assert bool((q[n:] == 0xA5).all())
    return q[:n], s[0]


def _check(lib, n, seed=1):
    x = torch.randn(n, device="cuda", generator=torch.Generator("cuda").manual_seed(seed))
    # The largest magnitude in turn in the first, a middle and the last element.
    for at in (0, n // 2 + 5, n - 1):
        x[at] = 9.0 + at % 3
        q, s = _run(lib, x, n)
        qw, sw = _want(x)
        assert s == sw and torch.equal(q, qw)
        x[at] = 0.5


# One more than a chunk per workgroup, whole and part chunks; all four held chunks of every
# workgroup, one less and one more; chunks read twice; then the two launches.
@pytest.mark.parametrize("n", [1024 * CHUNK + 1, 1025 * CHUNK, 1300 * CHUNK + 4099, 1536 * CHUNK - 2, 2048 * CHUNK,
                               2048 * CHUNK + 3, 2049 * CHUNK + 7, 2600 * CHUNK + 16383, 4097 * CHUNK,
                               16 * 512 * CHUNK + 5])
def test_sizes(lib, n):
    print(f"\n[quantize] n={n}", flush=True)
    _check(lib, n)


@pytest.mark.parametrize("n", [1100 * CHUNK + 9, 2100 * CHUNK])
def test_nan_and_fallback(lib, n):
    """A NaN anywhere makes every code NaN; with no polls allowed every workgroup finds the max
    itself, and the bits are the barrier's."""
    print(f"\n[quantize] NaN and fallback n={n}", flush=True)
    x = torch.randn(n, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    q0, s0 = _run(lib, x, n)
    hook = lib.taskops_testing_quantize_spin_limit
    hook.argtypes = [ctypes.c_uint]
    hook(0)
    try:
        q1, s1 = _run(lib, x, n)
    finally:
        hook(1 << 14)
    assert s0 == s1 and torch.equal(q0, q1)
    for at in (5, n - 1):
        x[at] = float("nan")
        q, s = _run(lib, x, n)
        assert bool(torch.isnan(s)) and bool(((q & 0x7F) == 0x7F).all())
        x[at] = 0.0


def test_graph_replay(lib):
    n = 1200 * CHUNK + 33
    print(f"\n[quantize] graph n={n}", flush=True)
    x = torch.randn(n, device="cuda")
    q = torch.zeros(n, dtype=torch.uint8, device="cuda")
    s = torch.zeros(1, device="cuda")
    args = dict(x=x, n=n, q=q, scale=s)
    capi.call(lib, "quantize_e4m3", args)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        capi.call(lib, "quantize_e4m3", args)
    for k in range(4):
        x.copy_(torch.randn(n, device="cuda") * (k + 1))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        qw, sw = _want(x)
        assert s[0] == sw and torch.equal(q, qw)


@pytest.mark.parametrize("n", [3, 16385, 5 * CHUNK + 1, 1024 * CHUNK, 1100 * CHUNK + 9, 2100 * CHUNK + 2, 4096 * CHUNK + 1])
def test_helping_and_alone(lib, n):
    """With no polls allowed the workgroups share out x among themselves; with none for the last
    pieces either, each may end up finding the max by itself.  Same bits, launch after launch,
    as the barrier's, with the largest magnitude in turn in the first and the last element."""
    print(f"\n[quantize] helping n={n}", flush=True)
    x = torch.randn(n, device="cuda", generator=torch.Generator("cuda").manual_seed(4))
    spin, wait = lib.taskops_testing_quantize_spin_limit, lib.taskops_testing_quantize_help_limit
    spin.argtypes = wait.argtypes = [ctypes.c_uint]
    try:
        for limits in [(0, 1 << 14), (0, 0), (1, 1 << 14), (0, 1 << 14)]:
            spin(limits[0])
            wait(limits[1])
            for at in (0, n - 1):
                x[at] = 9.0 + at % 3
                for _ in range(2):
                    q, s = _run(lib, x, n)
                    qw, sw = _want(x)
                    assert s == sw and torch.equal(q, qw), (limits, at)
                x[at] = 0.5
    finally:
        spin(128)
        wait(1 << 14)
    q, s = _run(lib, x, n)
    qw, sw = _want(x)
    assert s == sw and torch.equal(q, qw)


def test_beside_work_that_holds_the_chip(lib):
    """Elementwise kernels on another stream hold the CUs while tensors of every route are
    quantised: right codes, and no wait for a workgroup that is not running (16.8 M elements took
    9 ms when each waiting workgroup gave up on its own)."""
    print("\n[quantize] beside other work", flush=True)
    big = torch.randn(1 << 28, device="cuda")
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    for n in (1 << 24, 1 << 25, 1 << 26):
        x = torch.randn(n, device="cuda")
        qw, sw = _want(x)
        q = torch.zeros(n, dtype=torch.uint8, device="cuda")
        s = torch.zeros(1, device="cuda")
        torch.cuda.synchronize()
        took = []
        for _ in range(3):
            with torch.cuda.stream(s2):
                for _ in range(6):
                    big.mul_(1.0001)
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record(s1)
            capi.call(lib, "quantize_e4m3", dict(x=x, n=n, q=q, scale=s), s1.cuda_stream)
            b.record(s1)
            torch.cuda.synchronize()
            took.append(a.elapsed_time(b))
            assert s[0] == sw and torch.equal(q, qw)
        print(f"[quantize] n={n} {min(took):.3f} ms", flush=True)
        assert min(took) < 5.0
