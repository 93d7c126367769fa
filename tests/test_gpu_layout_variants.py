"""Block-size / scan-chunk library variants give the default build's
results bit for bit (the reductions add per-chunk partials whose grouping
changes with the block size, so this is a check, not a tautology): each
built variant steps a small DFSPH dam break in a process of its own (a
process loads one libsphg) and its final positions and iteration count are
compared with the default library's."""
import os
import subprocess
import sys

import pytest

from sph_amd import tune_layout

pytestmark = pytest.mark.gpu

VARIANTS = [(128, 1024), (512, 1024), (256, 256), (256, 4096)]


def test_layout_variants_match_default():
    built = [v for v in VARIANTS if os.path.exists(tune_layout.lib_path(*v))]
    if not built:
        pytest.skip("no layout variant is built (make -C sph_amd/csrc BLOCK=... CELL_CHUNK=...)")
    r = tune_layout.tune("dfsph_small", [tune_layout.DEFAULT] + built, timeout=120.0, log=lambda s: None)
    rows = {(x["block"], x["scan_chunk"]): x for x in r["variants"]}
    ref = rows[tune_layout.DEFAULT]
    for v in built:
        assert rows[v]["x_max_diff_vs_default"] == 0.0, (v, rows[v])
        assert rows[v]["density_iterations"] == ref["density_iterations"], (v, rows[v])


CHILD = """
import sys
import numpy as np
from sph_amd import configs, sphg
sphg.load(sys.argv[1])
ctx = sphg.Context(0)
spec = configs.small_scene(sphg.DFSPH, n_side=31)
other = configs.small_scene(sphg.DFSPH, n_side=5)
v = np.random.default_rng(5).uniform(-1, 1, spec.fluid.shape).astype(np.float32)
alone, mixed = [sphg.Scene(ctx, spec.params, spec.fluid, spec.boundary, v) for _ in range(2)]
extra = sphg.Scene(ctx, other.params, other.fluid, other.boundary)
for step in range(12):
    alone.step(1)
    ctx.batch_step([mixed, extra], 1)
    a, m = alone.scalars(), mixed.scalars()
    for name, _ in a._fields_:
        assert getattr(a, name) == getattr(m, name), (step, name, getattr(a, name), getattr(m, name))
assert np.array_equal(alone.get(sphg.FIELD_X), mixed.get(sphg.FIELD_X))
"""


@pytest.mark.parametrize("variant", VARIANTS)
def test_layout_variant_alone_and_in_a_batch(variant):
    """The error sums that decide a loop are added in one order, whether the
    sweeps of a lone scene or the finalize kernels of a batch form them, also
    where a chunk is not the 256 threads of the sweeps with 4 lanes a
    particle (29,791 particles: 233 partials with blocks of 128)."""
    lib = tune_layout.lib_path(*variant)
    if not os.path.exists(lib):
        pytest.skip("the layout variant is not built (make -C sph_amd/csrc BLOCK=... CELL_CHUNK=...)")
    r = subprocess.run([sys.executable, "-c", CHILD, lib], capture_output=True, text=True, timeout=100,
                       cwd=os.path.dirname(tune_layout.HERE))
    assert r.returncode == 0, r.stderr[-2000:]
