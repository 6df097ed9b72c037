"""The default kernel form by view (images.py:30-144 of the reference): up to
|a sin i| = 0.5 by the tile count alone, beyond it the triple form for larger
launches too; and for larger ones the wider the field of view.  The image is the
same bits whichever form runs."""
import ctypes as C

import numpy as np
import pytest

from mahakala_amd import _lib, images
from mahakala_amd.grmhd import synthetic as syn
from mahakala_amd.grmhd.athenak import AthenakFluidModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,spin,inc,res,form", [
    ("mixed", 0.5, 85.0, 512, "classic"), ("plain64", 0.5, 85.0, 440, "classic"),  # |a sin i| just below 0.5
    ("mixed", 0.51, 85.0, 512, "triple"), ("plain64", -0.51, 85.0, 440, "triple"),  # and just above
    ("mixed", 0.95, 20.0, 512, "classic"), ("mixed", 0.9, 60.0, 640, "triple"), ("plain64", 0.7, 50.0, 576, "classic"),
])
def test_default_form_and_image(precision, spin, inc, res, form):
    m = AthenakFluidModel.from_datasets(syn.uniform_torus_snapshot(spin, seed=0), spin, fluid_gamma=13. / 9)
    out = {}
    for f in (None, "classic", "triple"):
        p = images.render_params(spin, camera_inclination=inc, resolution=res, precision=precision, form=f)
        got = C.c_int32()
        _lib.check(_lib.lib().mk_render_form(m.device_snapshot.handle, p, C.byref(got)))
        assert got.value == images.FORMS[form if f is None else f]
        out[f] = images.render(m.device_snapshot, p)
    np.testing.assert_array_equal(out[None], out["classic"])
    np.testing.assert_array_equal(out[None], out["triple"])


@pytest.mark.parametrize("precision,spin,inc,fov,res,form", [
    ("mixed", 0.0, 45.0, 60.0, 640, "triple"), ("mixed", 0.0, 45.0, 60.0, 704, "classic"), ("plain64", 0.0, 45.0, 60.0, 560, "triple"),
    ("mixed", 0.9, 60.0, 12.0, 656, "triple"), ("mixed", 0.9, 60.0, 12.0, 768, "classic"), ("mixed", 0.5, 30.0, 12.0, 464, "classic"),
    ("plain64", 0.5, 30.0, 8.0, 352, "classic"), ("mixed", -0.97, 85.0, 36.0, 1024, "triple"), ("mixed", 0.0, 45.0, 300.0, 768, "triple"),
])
def test_default_form_by_field_of_view(precision, spin, inc, fov, res, form):
    """On the GPU's 256 CUs; the lines lie between the sizes."""
    m = AthenakFluidModel.from_datasets(syn.uniform_torus_snapshot(0.5, seed=0, nblocks=4, n=16), 0.5, fluid_gamma=13. / 9)
    out = {}
    for f in (None, "classic", "triple"):
        p = images.render_params(spin, camera_inclination=inc, resolution=res, fov=fov, precision=precision, form=f)
        got = C.c_int32()
        _lib.check(_lib.lib().mk_render_form(m.device_snapshot.handle, p, C.byref(got)))
        assert got.value == images.FORMS[form if f is None else f]
        out[f] = images.render(m.device_snapshot, p)
    np.testing.assert_array_equal(out[None], out["classic"])
    np.testing.assert_array_equal(out[None], out["triple"])
