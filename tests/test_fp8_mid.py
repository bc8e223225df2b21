"""fp8_linear's middle kernel (64x64, 64x128 and 128x128 tiles, any K and alignment) at the edges
of its tiles, steps and 16-byte loads, and the 128x256 form's tails at the sizes that still take
it, against the fp64 oracle at the task tolerance (atol = rtol = 1e-2, one bf16 rounding)."""
import numpy as np
import pytest
import torch

from cob_amd import capi, inputs, tasks
from cob_amd.grader.tolerance import tally
from oracle import exact

pytestmark = pytest.mark.gpu

# (M, K, N, operand offset in bytes, output offset in elements)
SHAPES = [
    # 64x64 tiles, direct copies: one tile and ragged ones, one step to more than the ring holds
    (65, 16, 64, 0, 0), (64, 128, 65, 0, 0), (128, 144, 63, 0, 0), (100, 512, 200, 0, 0), (127, 1040, 130, 0, 4),
    (33, 640, 72, 0, 1), (48, 656, 1, 0, 0), (16, 256, 8192, 0, 0), (32, 272, 5121, 0, 0),
    # at most 64 rows: few columns and K past 2048, more than 16 columns per CU, and the ring of 8
    # steps (up to 32 rows, K from 4096 on) with ragged tails
    (33, 2064, 520, 0, 0), (48, 3088, 1000, 0, 1), (40, 4096, 515, 0, 0), (64, 4112, 70, 0, 0), (40, 144, 4100, 0, 0), (64, 528, 4225, 0, 0),
    (16, 4096, 7168, 0, 0), (1, 4112, 7201, 0, 0), (17, 4224, 5125, 0, 0), (32, 4240, 5120, 0, 4),
    # 64x128 and 128x128 tiles, direct copies
    (513, 400, 4000, 0, 0), (400, 768, 4100, 0, 0), (1000, 912, 4100, 0, 0), (777, 1024, 4001, 0, 3),
    # 16-byte loads at any alignment: K below 16, on both sides of a load and of a step
    (65, 1, 64, 0, 0), (70, 7, 33, 0, 0), (5, 15, 40, 0, 0), (66, 17, 64, 0, 0), (1, 31, 65, 0, 0), (80, 33, 70, 0, 0),
    (130, 127, 64, 0, 0), (64, 129, 128, 0, 0), (90, 130, 96, 0, 0), (67, 255, 31, 0, 0), (200, 257, 300, 0, 0),
    (333, 1000, 3000, 0, 0), (600, 143, 3001, 0, 0), (1500, 72, 2999, 0, 0), (1100, 388, 4096, 0, 0), (12, 999, 301, 0, 1),
    (50, 520, 4200, 0, 0),
    # K % 16 == 0 at unaligned operands
    (100, 256, 72, 1, 0), (100, 256, 72, 4, 0), (20, 256, 72, 2, 0), (300, 64, 300, 8, 0),
    # 128x256 tiles (half) with each epilogue and ragged tails
    (2000, 144, 4000, 0, 0), (2000, 144, 4004, 0, 4), (1990, 176, 3999, 0, 0),
]


@pytest.mark.parametrize("M,K,N,off,oout", SHAPES)
def test_shapes(lib, M, K, N, off, oout):
    print(f"\n[fp8_mid] M{M} K{K} N{N} offset {off}/{oout}", flush=True)
    inp = inputs.make_inputs("fp8_linear", dict(name="f", seed=800 + M + K + N, M=M, K=K, N=N))
    args = capi.device_args("fp8_linear", inp)
    for name in ("x_fp8", "w_fp8"):
        t = torch.full((args[name].numel() + off,), 0x7F, dtype=torch.uint8, device="cuda")  # NaN before the operand
        t[off:] = args[name].flatten()
        args[name] = t[off:]
    out = torch.full((M * N + oout + 64,), float("nan"), dtype=torch.bfloat16, device="cuda")
    args["output"] = out[oout:]
    capi.call(lib, "fp8_linear", args)
    torch.cuda.synchronize()
    first = out.clone()
    capi.call(lib, "fp8_linear", args)
    torch.cuda.synchronize()
    assert torch.equal(first.view(torch.int16), out.view(torch.int16))
    got = out[oout:oout + M * N].reshape(M, N).float().cpu().numpy()
    t = tally(got, exact.fp8_linear(inp)["output"], tasks.load_task("fp8_linear")["tolerance"])
    assert t["mismatched"] == 0, t
    assert bool(torch.isnan(out[:oout].float()).all()) and bool(torch.isnan(out[oout + M * N:].float()).all())


@pytest.mark.parametrize("M,K,N", [(100, 256, 72), (70, 1001, 33), (600, 300, 3000), (65, 9, 20)])
def test_special_codes(lib, M, K, N):
    """A NaN in one row of x reaches that row alone, also in a K tail; zero x gives the bias."""
    print(f"\n[fp8_mid] codes M{M} K{K} N{N}", flush=True)
    inp = inputs.make_inputs("fp8_linear", dict(name="f", seed=9, M=M, K=K, N=N))
    xb = torch.zeros(M, K, dtype=torch.uint8)
    xb[3, K - 1] = 0x7F
    xb[M - 1, 0] = 0xFF
    inp["x_fp8"] = xb.view(torch.float8_e4m3fn)
    got = capi.run_op(lib, "fp8_linear", inp)["output"].cpu()
    keep = [r for r in range(M) if r not in (3, M - 1)]
    assert torch.isnan(got[3].float()).all() and torch.isnan(got[M - 1].float()).all()
    assert np.array_equal(got[keep].float().numpy(), inp["bias"].float().reshape(1, N).expand(len(keep), N).numpy())
