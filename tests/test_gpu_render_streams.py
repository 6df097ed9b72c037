"""mk_render from several streams (images.py:30-144 of the reference): a view's
tile order is built by its first launch and read by every later one, on
whichever stream."""
import pytest
import torch

from mahakala_amd import _lib, images
from mahakala_amd.grmhd import synthetic as syn
from mahakala_amd.grmhd.athenak import AthenakFluidModel

pytestmark = pytest.mark.gpu
ROW_MAJOR = 512  # MK_RENDER_ROW_MAJOR


@pytest.mark.parametrize("form,res", [(None, 272), ("classic", 304), ("triple", 336)])
def test_first_view_on_a_busy_stream_and_again_on_another(form, res):
    m = AthenakFluidModel.from_datasets(syn.uniform_torus_snapshot(0.5, seed=0, nblocks=4, n=16), 0.5, fluid_gamma=13. / 9)
    p = images.render_params(0.5, camera_inclination=41.375, resolution=res, precision="mixed", form=form)
    ref, a, b = (torch.zeros((res, res), device="cuda", dtype=torch.float64) for _ in range(3))
    lib, snap = _lib.lib(), m.device_snapshot.handle
    p.flags |= ROW_MAJOR
    _lib.check(lib.mk_render(snap, p, ref.data_ptr(), None, None))
    p.flags &= ~ROW_MAJOR
    x = torch.ones((8192, 8192), device="cuda", dtype=torch.bfloat16)
    torch.cuda.synchronize()
    busy, other = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(busy):
        for _ in range(60):
            y = x @ x
    _lib.check(lib.mk_render(snap, p, a.data_ptr(), None, busy.cuda_stream))
    held = not busy.query()  # the first launch still waits behind the products
    _lib.check(lib.mk_render(snap, p, b.data_ptr(), None, other.cuda_stream))
    other.synchronize()
    assert torch.equal(b, ref)
    busy.synchronize()
    assert torch.equal(a, ref)
    assert held and y is not None
