"""Image-only launches of the persistent server: four waves per tile, or one
wave per tile when the launch starts with a deep backlog (images.py:30-144 of
the reference).  Both give mk_render's bits, whatever the tile count."""
import ctypes as C
import time

import numpy as np
import pytest

import mahakala_amd as ma
from mahakala_amd import _lib, images
from mahakala_amd.constants import Msun
from mahakala_amd.grmhd import synthetic as syn
from mahakala_amd.grmhd.athenak import AthenakFluidModel
from mahakala_amd.serving import Server

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model():
    return AthenakFluidModel.from_datasets(syn.uniform_torus_snapshot(0.9, seed=0), 0.9, fluid_gamma=13. / 9)


def _render(model, view, precision):
    p = images.render_params(0.9, camera_inclination=view["inclination"], resolution=view["resolution"], fov=20,
                             observing_frequency=230e9, max_nsteps=view["max_nsteps"], precision=precision)
    return images.render(model.device_snapshot, p)


def _submit(srv, sid, view):
    return srv.submit_image(sid, bhspin=0.9, observing_frequency=230e9, fov=20, **view)


@pytest.mark.parametrize("precision", ["plain64", "mixed"])
def test_tiles_of_any_count_and_step_limit(model, precision):
    views = [dict(resolution=r, inclination=i, max_nsteps=n)
             for r, i, n in [(1, 30.0, 10000), (7, 60.0, 10000), (8, 60.0, 10000), (9, 85.0, 300), (36, 10.0, 1),
                             (64, 75.0, 10000), (65, 5.0, 90)]]
    with Server(precision, lanes=1024, image_in_launch=True) as srv:
        sid = srv.add_snapshot(model)
        for _ in range(2):  # the second pass reuses the request slots
            rids = [_submit(srv, sid, v) for v in views]
            for v, rid in zip(views, rids):
                np.testing.assert_array_equal(srv.result(rid, timeout=60), _render(model, v, precision), err_msg=str(v))


@pytest.mark.parametrize("precision", ["plain64", "mixed"])
def test_deep_backlog_behind_a_shallow_launch(model, precision):
    """At 2048 lanes 8192 items make a launch start deep and 32768 end a
    shallow one: 48^2 starts shallow, 12 images of 64^2 follow it."""
    first = dict(resolution=48, inclination=60.0, max_nsteps=10000)
    later = [dict(resolution=64, inclination=5.0 + 6 * k, max_nsteps=10000) for k in range(12)]
    with Server(precision, lanes=2048, image_in_launch=True) as srv:
        sid = srv.add_snapshot(model)
        rids = [_submit(srv, sid, first)]
        t_wait = time.perf_counter() + 30.0
        while srv.stats()["iterations"] < 1:
            assert time.perf_counter() < t_wait, "the first launch did not start"
            time.sleep(0.0005)
        rids += [_submit(srv, sid, v) for v in later]
        got = [srv.result(r, timeout=60) for r in rids]
        time.sleep(0.1)  # longer than the idle limit: the launch ends
        st = srv.stats()
    assert st["completed"] == 13 and st["in_flight"] == 0 and st["iterations"] >= 2
    for v, img in zip([first] + later, got):
        np.testing.assert_array_equal(img, _render(model, v, precision), err_msg=str(v))


@pytest.mark.parametrize("precision", [0, 1])
def test_a_tile_whose_waves_gave_up_does_not_complete_its_request(model, precision):
    """With a limit of one poll the waves of a tile give up on each other: the
    server reports it, and no request is handed out as completed with the NaN of
    such a tile."""
    lib, n = _lib.lib(), 64
    cfg = _lib.mk_server_config(precision, 0, 0, 0, 0, 0, 1 | 4 | 8)  # PERSISTENT, IMAGE_IN_LAUNCH, WAIT_TEST
    h, sid, rid = _lib.vp(), C.c_int32(), C.c_int64()
    _lib.check(lib.mk_server_create(C.byref(cfg), C.byref(h)))
    try:
        _lib.check(lib.mk_server_add_snapshot(h, model.device_snapshot.handle, C.byref(sid)))
        out = np.full((n, 16, 16), -7.0)
        ids = []
        for k in range(n):
            req = _lib.mk_image_request(sid.value, 16, 10000, 0, 0.9, 30.0 + k / 4, 1000.0, 10.0, 230e9, 1e26, 6.2e9 * Msun,
                                        40.0, 13. / 9)
            if lib.mk_server_submit_image(h, C.byref(req), out[k].ctypes.data, C.byref(rid)):
                break  # the error is out already
            ids.append(rid.value)
        assert ids
        assert {lib.mk_server_wait(h, i, 30.0) for i in ids + [-1]} == {-5}  # MK_ERR_STATE
        assert b"waited longer than its limit" in lib.mk_last_error()
        st = _lib.mk_server_stats()
        assert lib.mk_server_get_stats(h, C.byref(st)) == -5  # filled in all the same
        assert st.completed == 0 and (out == -7.0).all()
    finally:
        _lib.check(lib.mk_server_destroy(h))


@pytest.mark.parametrize("shadows", [False, True])
def test_many_requests_published_together(model, shadows):
    """Requests of one published batch share a copy to device memory: small and
    large tile orders, images without one (size not a multiple of 8), one too long
    to be copied, and bisections between them, behind an image that keeps the
    launch busy while they gather."""
    sizes = [256] + [8, 16, 8, 33, 64, 8, 8, 7, 24, 8, 8, 8, 8, 8, 8, 8, 8, 8, 8, 128, 160, 9, 16, 8, 1032, 8, 48] * 2 + [8] * 70
    views = [dict(resolution=r, inclination=5.0 + (7 * k) % 80, max_nsteps=10000 if r < 1000 else 340)
             for k, r in enumerate(sizes)]
    ang = np.arange(5.0)
    with Server("mixed", image_in_launch=True, shadow_in_launch=True) as srv:
        sid = srv.add_snapshot(model)
        for _ in range(2):
            rids = []
            for k, v in enumerate(views):
                rids.append(_submit(srv, sid, v))
                if shadows and k % 11 == 0:
                    rids.append(srv.submit_shadow(0.9, 60.0, ang + k, max_steps=50))
            got = [srv.result(r, timeout=60) for r in rids]
    images_got = [g for g in got if g.ndim == 2]
    for v, img in zip(views, images_got):
        np.testing.assert_array_equal(img, _render(model, v, "mixed"), err_msg=str(v))
    if shadows:
        want = [ma.find_shadow_bisection_angles(0.9, 60.0, ang + k, max_steps=50) for k in range(0, len(views), 11)]
        np.testing.assert_array_equal([g for g in got if g.ndim == 1], want)
