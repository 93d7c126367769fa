"""A step's launch variants give one result: what a rule on sizes, options or
the launch's scenes picks between must not change a bit of it."""
import numpy as np
import pytest

from sph_amd import configs, sphg

pytestmark = pytest.mark.gpu

METHODS = [sphg.WCSPH, sphg.PCISPH, sphg.DFSPH]
FORCES = {
    "none": {},
    "xsph": dict(viscosity_method=sphg.VISCOSITY_XSPH, viscosity=0.02, boundary_viscosity=0.01),
    "cohesion": dict(surface_tension_method=sphg.SURFACE_TENSION_AKINCI, surface_tension=0.05),
    "adhesion": dict(adhesion_method=sphg.ADHESION_AKINCI, adhesion=0.1),
    "standard": dict(viscosity_method=sphg.VISCOSITY_STANDARD, viscosity=0.01),
}
FORCES["xsph_cohesion"] = {**FORCES["xsph"], **FORCES["cohesion"]}
FORCES["all"] = {**FORCES["xsph_cohesion"], **FORCES["adhesion"]}


def fields(scene):
    out = [scene.get(sphg.FIELD_X), scene.get(sphg.FIELD_V), scene.get(sphg.FIELD_A), scene.get(sphg.FIELD_DRHO)]
    if scene.params.method == sphg.DFSPH:
        out += [scene.get(sphg.FIELD_K), scene.get(sphg.FIELD_KV)]
    return out


def same(a, b):
    return all(np.array_equal(x, y, equal_nan=True) for x, y in zip(fields(a), fields(b)))


@pytest.mark.parametrize("method", METHODS)
@pytest.mark.parametrize("forces", sorted(FORCES))
def test_forces_kernel_of_one_and_of_mixed_options(ctx, method, forces):
    """Alone, a scene's forces run in the kernel compiled for its options; in
    a batch with a scene of other options, in the general one.  The ragged
    size leaves the last wavefront partly empty."""
    other = "standard" if forces != "standard" else "xsph"
    specs = [configs.small_scene(method, n_side=(9, 7, 8), box=(1.2, 0.55, 0.8), **FORCES[f]) for f in (forces, other)]
    alone, mixed, extra = [sphg.Scene(ctx, s.params, s.fluid, s.boundary) for s in (specs[0], specs[0], specs[1])]
    alone.step(4)
    ctx.batch_step([mixed, extra], 4)
    assert same(alone, mixed)
    for s in (alone, mixed, extra):
        s.close()
