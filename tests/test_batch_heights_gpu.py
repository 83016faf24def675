"""Segment heights of a batch of mixed sizes: its longest item ends a pass."""

import math
import random

import pytest
import torch

import perks_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", ["2d5pt", "2d9pt"])
@pytest.mark.parametrize("seed", [0, 512])
def test_mixed_sizes_fill_the_chip(shape, seed):
    """512 grids of 64 to 1024 a side hold some 250 rows for every wave that the
    chip can run at once, so no height that leaves one of four waves per SIMD out
    (the tall grids cut into few long items) is the shortest pass."""
    rng = random.Random(seed)

    def side():
        return round(math.exp(rng.uniform(math.log(64), math.log(1024))))

    dims = [(side(), side(), rng.randint(50, 500)) for _ in range(512)]
    a = torch.rand(sum(h * w for h, w, _ in dims), device="cuda")
    b = torch.zeros_like(a)
    grids, at = [], 0
    for h, w, steps in dims:
        grids.append((a[at : at + h * w], b[at : at + h * w], h, w, steps))
        at += h * w
    points = 5 if shape == "2d5pt" else 9
    opts = P.make_opts(shape, "zero", "persistent", coefs=[1 / points] * len(P.shape_info(shape).coef))
    plan = P.BatchPlan(grids, dtype="f32", autotune=False, opts=opts)
    try:
        assert plan.config["workgroups"] >= 4 * torch.cuda.get_device_properties(0).multi_processor_count
    finally:
        plan.close()
