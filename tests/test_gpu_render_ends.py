"""Where a ray of the image kernel may end (images.py:30-144 of the reference).

Without step counts a ray ends once it has left the sphere around the domain
outward, and the triple form hands no sample over before a ray of its tile
enters that sphere.  Neither changes a bit of the image: the launch that
returns step counts follows every ray to its end.
"""
import numpy as np
import pytest

from mahakala_amd import images
from mahakala_amd.grmhd import synthetic as syn
from mahakala_amd.grmhd.athenak import AthenakFluidModel

pytestmark = pytest.mark.gpu


def _model(spin, extent, offset=0.0):
    """The torus on 2^3 blocks of 8^3 cells over [-extent, extent]^3, shifted by `offset` along x."""
    geo = syn.uniform_layout(extent=extent, nblocks=2, n=8)
    geo["x1f"], geo["x1v"] = geo["x1f"] + np.float32(offset), geo["x1v"] + np.float32(offset)
    x, y, z = np.broadcast_arrays(geo["x1v"][:, None, None, :], geo["x2v"][:, None, :, None],
                                  geo["x3v"][:, :, None, None])
    f = syn.torus_fields(x, y, z, spin)
    ds = {k: geo[k] for k in ("x1v", "x2v", "x3v", "x1f", "x2f", "x3f", "Levels", "LogicalLocations")}
    ds.update(uov=np.stack([f[k] for k in ("dens", "velx", "vely", "velz", "u")]),
              B=np.stack([f[k] for k in ("bcc1", "bcc2", "bcc3")]), VariableNames=list(syn.VARIABLE_NAMES))
    return AthenakFluidModel.from_datasets(ds, spin, fluid_gamma=13. / 9)


@pytest.mark.parametrize("precision", ["plain64", "mixed", "mixed-zone"])
@pytest.mark.parametrize("extent,offset,view", [
    (40.0, 0.0, dict(fov=20)),                                # the usual view; 13^2 leaves partial tiles
    (40.0, 0.0, dict(fov=20, camera_distance=30)),            # the camera inside the domain
    (5.0, 0.0, dict(fov=16)),                                 # a domain that ends near the photon orbits
    (40.0, 30.0, dict(fov=60)),                               # a domain off the hole's centre
    (40.0, 0.0, dict(fov=400)),                               # most rays never enter
    (40.0, 0.0, dict(fov=20, max_nsteps=90)),                 # cut on the way in,
    (40.0, 0.0, dict(fov=20, max_nsteps=300)),                # inside
    (40.0, 0.0, dict(fov=20, max_nsteps=1)),                  # and at the first step
])
def test_image_is_the_same_with_and_without_step_counts(precision, extent, offset, view):
    m = _model(0.9, extent, offset)
    for form in ("triple", "classic", "paired", None):
        p = images.render_params(0.9, camera_inclination=50, resolution=13, precision=precision, form=form, **view)
        if precision == "mixed-zone":
            p.fp64_radius = 100.0  # a zone larger than the domain: its rays decide the tile's FP64 steps
        whole, steps = images.render(m.device_snapshot, p, return_steps=True)
        assert steps.max() > 0 or view.get("max_nsteps") == 1
        np.testing.assert_array_equal(images.render(m.device_snapshot, p), whole)
        if form == "triple":
            first = whole
        np.testing.assert_array_equal(whole, first)
