"""What the trained pre-sizer gains over the method without it.

The first 65,536 paths of the pre-sizer's evaluation scene (outlines of the
uneven family on 8192^2) are drawn four ways: by the exact two-pass method
(count passes, read-back, write passes), by the exact method as it draws by
default (planes for every tile reserved instead of counted, where that fits), by
the learned single-pass method (the MLP's capacities, fallback to the exact
method on under-prediction) and by the same single-pass method with capacities
from a bound linear in the segment count and the bounding box (no network).
The four frames must be identical; the learned form must be faster than the
two-pass method, whose count pass it saves.  The default exact form saves it as
well and is as fast as the learned one here (0.99 to 1.01 of its time over six
runs), so that is reported and not asserted, as is the linear row.
"""
import numpy as np
import pytest

from skity_amd import device, presizer

pytestmark = pytest.mark.gpu


def test_learned_presizing_gain_at_identical_output():
    ctx = device.Context(0)
    try:
        presizer.install(ctx, *presizer.load())
        # one warm-up slice so first-use allocations are not timed
        presizer.evaluate_large(ctx, n_paths=4096, slice_paths=4096, log=lambda m: None)
        rep = presizer.evaluate_large(ctx, n_paths=65536, slice_paths=65536,
                                      log=lambda m: print(m, flush=True))
    finally:
        ctx.close()
    for k in ("exact", "two_pass", "learned", "linear_estimate"):
        r = rep[k]
        print(f"{k}: {r['ms']:.1f} ms, {r['paths_per_s']:.0f} paths/s, fallback rate "
              f"{r['fallback_rate']:.4f}, under-estimate rate {r['underestimate_rate']:.4f}, "
              f"identical {r['identical_to_exact']}", flush=True)
    assert rep["two_pass"]["identical_to_exact"]
    assert rep["learned"]["identical_to_exact"]
    assert rep["linear_estimate"]["identical_to_exact"]
    assert rep["learned"]["jobs"] == rep["exact"]["jobs"] > 60000
    assert "walk_count" in rep["two_pass"]["stage_ms"]
    assert "walk_count" not in rep["exact"]["stage_ms"]
    gain = rep["two_pass"]["ms"] / rep["learned"]["ms"]
    print(f"learned vs two-pass: {gain:.2f}x; vs exact: "
          f"{rep['exact']['ms'] / rep['learned']['ms']:.2f}x; linear estimate vs two-pass: "
          f"{rep['two_pass']['ms'] / rep['linear_estimate']['ms']:.2f}x", flush=True)
    assert gain > 1.0
    assert rep["learned"]["fallback_rate"] < 0.05
