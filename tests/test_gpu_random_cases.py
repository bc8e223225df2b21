"""Seeded random shapes for every op through the three-call protocol on guarded device arenas.

The reference grader's checks, per case: every output within the task tolerance of
reference_exact on calls 1 and 3, nothing written outside the outputs, inputs untouched, and
identical bits on the repeated inputs (graders/child.py:141-204).  The fixed shape lists in
test_gpu_parity.py sit on each kernel's boundaries (tile tails, chunk counts, launch shapes);
these cases draw shapes between and across them, with the distribution parameters the input
builders take (scale, mem0, beta range, gamma, done rate, clip epsilon, knot count and
spline order, x range).  fp8_linear's K includes values off a multiple of 16, which take the
register-staged and byte-wise loads.  efficient_kan's draws are small and take its direct path;
a second set has the batches and widths of the packed one (test_host_paths.py pins that).  The draws are fixed by the seed below, so a failure
names a reproducible case.
"""
import random

import pytest

from cob_amd import tasks
from cob_amd.grader.labels import kernel_status
from cob_amd.grader.protocol import run_case
from oracle import exact

pytestmark = pytest.mark.gpu

SEED = 20261202
PER_OP = 24


def _draw(op: str, rng: random.Random, i: int) -> dict:
    c = {"name": f"rand{i}", "seed": 90_000 + 97 * i + 7 * tasks.OPS.index(op), "small": False, "timed": False}
    if op == "pow_abs_sqrt_mean":
        c.update(batch_size=rng.randint(1, 6), height=rng.randint(1, 160), width=rng.randint(1, 160),
                 scale=rng.choice([1.0, 1.0, 1000.0]))
    elif op == "leaky":
        c.update(T=rng.randint(1, 48), B=rng.randint(1, 40), H=rng.randint(1, 300),
                 mem0_std=rng.choice([0.0, 0.5]), beta_range=rng.choice([[0.65, 0.98], [-0.2, 1.3]]))
    elif op == "reward_to_go":
        c.update(B=rng.randint(1, 40), T=rng.randint(1, 5000), gamma=rng.uniform(0.8, 1.0),
                 done_p=rng.choice([0.0, 0.01, 0.1, 0.5]))
    elif op == "ppo_clip":
        c.update(B=rng.randint(1, 8), T=rng.randint(1, 300), H=rng.randint(1, 20),
                 clip_epsilon=rng.uniform(0.05, 0.4), delta_std=rng.choice([0.01, 0.12, 1.0]))
    elif op == "efficient_kan":
        k = rng.randint(1, 4)
        c.update(B=rng.randint(1, 300), I=rng.randint(1, 150), O=rng.randint(1, 300),
                 grid_size=rng.randint(1, 12), spline_order=k if rng.random() < 0.5 else 3,
                 x_range=rng.uniform(0.5, 1.5))
    elif op == "fp8_linear":
        K = rng.choice([rng.randint(1, 1500), 16 * rng.randint(1, 96)])
        c.update(M=rng.choice([rng.randint(1, 64), rng.randint(65, 700)]), K=K, N=rng.randint(1, 700))
    return c


def _cases():
    rng = random.Random(SEED)
    return [(op, _draw(op, rng, i)) for op in tasks.OPS for i in range(PER_OP)]


def _packed_cases(n=8):
    """efficient_kan cases of the packed path: order 3, at most 16 knots."""
    rng = random.Random(SEED + 1)
    return [("efficient_kan", {"name": f"packed{i}", "seed": 97_000 + 31 * i, "small": False, "timed": False,
                               "B": rng.randint(3000, 6000), "I": rng.randint(64, 200), "O": rng.randint(513, 768),
                               "grid_size": rng.randint(1, 9), "spline_order": 3, "x_range": rng.uniform(0.5, 1.5)})
            for i in range(n)]


PACKED_CASES = _packed_cases()
CASES = _cases() + PACKED_CASES


def _label(c: dict) -> str:
    keys = [k for k in c if k not in ("name", "seed", "small", "timed")]
    return c["name"] + "_" + "_".join(f"{k}{c[k]:.3g}" if isinstance(c[k], float) else f"{k}{c[k]}"
                                      for k in keys if not isinstance(c[k], list))


@pytest.mark.parametrize("op,case", CASES, ids=[f"{op}-{_label(c)}" for op, c in CASES])
def test_random_case_three_call_protocol(lib, op, case):
    print(f"\n[random] {op} {_label(case)}", flush=True)
    report = run_case(op, case, exact.reference_exact)
    st = kernel_status([[report]])
    assert st["status"] == "pass", (st, report.get("checks"), report.get("calls"))
    assert report["repeat_identical"]
