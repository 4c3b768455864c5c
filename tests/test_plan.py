"""The forward's plans (moe.c, built for the CPU by tests/plan_scan.c) over
shapes and token counts: what a plan may not do, whatever it is chosen for."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    exe = tmp_path_factory.mktemp("plan") / "plan_scan"
    cmd = ["gcc", "-std=gnu99", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-no-pie",
           "-Wl,--unresolved-symbols=ignore-all", "-o", str(exe),
           os.path.join(ROOT, "tests", "plan_scan.c"), "-lm"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]

    def run(cases):
        text = "\n".join(" ".join(map(str, c)) for c in cases)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True,
                             timeout=300).stdout
        return np.array([line.split() for line in out.splitlines()], int)
    return run


def shapes(rng, n):
    E = rng.integers(1, 257, n)
    k = np.minimum(rng.integers(1, 17, n), E)
    T = np.exp(rng.uniform(0, np.log(4096), n)).astype(int)
    return np.stack([rng.integers(0, 3, n), rng.choice([256, 512, 1024, 2048, 4096], n),
                     rng.choice([256, 512, 1024], n), E, k, rng.integers(0, 2, n),
                     rng.integers(0, 2, n), T], axis=1)


def test_what_fits_the_fixed_scratch_is_not_refused(plans):
    """No call is refused by gpu_moe_forward_noalloc for the plan it got where
    another plan of the same products would fit."""
    cases = shapes(np.random.default_rng(1), 200_000)
    cases[0] = (0, 4096, 1024, 52, 2, 0, 0, 417)  # four tiles fit, two do not
    cases[1] = (0, 2048, 512, 112, 15, 0, 0, 121)
    got = plans(cases)
    lost = cases[(got[:, 4] == 0) & (got[:, 5] == 1)]
    assert not len(lost), lost[:10]
    assert (got[:2, 4] == 1).all()


def test_gate_up_slices_of_thin_batches(plans):
    """Up to 16 rows per expert a gate/up sum is at most 16 steps (512
    products) long, unless the shape has no shorter slice."""
    cases = shapes(np.random.default_rng(2), 100_000)
    cases[:, 0] = 0
    got = plans(cases)
    T, E, k, D = (cases[:, i] for i in (7, 3, 4, 1))
    thin = (got[:, 0] == 1) & (T * k <= 16 * E)
    assert thin.sum() > 10_000
    steps = D // 32 // got[:, 2]
    assert (steps[thin] <= 16).all(), cases[thin][steps[thin] > 16][:10]


def test_router_kernels_by_their_work():
    """The routing kernels are chosen by the work groups they have (tokens times
    experts), so that a layer of fewer experts keeps the faster ones to more
    tokens: the one-token-per-group router up to 1536 groups of eight experts
    (with the norm inside 2048, 1152 or 1024 by the width), one token per wave
    as long as four times the experts take a quarter of the tokens."""
    import ornith_moe
    pc, tpw = ornith_moe.lib().ornk_router_pc_supported, ornith_moe.lib().ornk_router_tpw
    for D, norm, most in ((256, 0, 1536), (2048, 0, 1536), (4096, 0, 1536), (1024, 1, 2048),
                          (2048, 1, 1152), (4096, 1, 1024)):
        for E in (8, 64, 128, 256):
            assert pc(8 * most // E, E, D, norm) and not pc(8 * most // E + 1, E, D, norm)
        assert pc(most // 2, 9, D, norm) and not pc(most // 2 + 1, 9, D, norm)
    for T in (4, 500, 640, 641, 1536, 1537, 4096):
        assert tpw(T, 256) == tpw(2 * T, 128) == tpw(4 * T, 64) == tpw(4 * T, 8)
