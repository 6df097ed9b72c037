"""Lanes without a ray of their own (geodesics.py:291-435 of the reference).

The FP64 walks keep every lane of a wave stepping, also those whose ray has
ended and those past the last ray: a ray's results do not depend on how many
others share its wave, and nothing is written past the last one.  The
bisection's schedule (lanes per angle, width of the band, angles per wave)
changes no radius.
"""
import ctypes as C

import numpy as np
import pytest
import torch

import mahakala_amd as ma
from mahakala_amd import _lib
from oracle import c_oracle

pytestmark = pytest.mark.gpu
GUARD = -7.0


def _start(n):
    s = torch.empty((12 * 12, 8), device="cuda", dtype=torch.float64)
    _lib.check(_lib.lib().mk_camera_grid(0.9, 60.0, 1000.0, -10.0, 10.0, 12, s.data_ptr(), None))
    return s[torch.arange(n, device="cuda") % 144].contiguous()


def _final(s0, N):
    n = len(s0)
    K = torch.full((n + 2,), -7, device="cuda", dtype=torch.int32)
    last = torch.full((n + 2, 8), GUARD, device="cuda", dtype=torch.float64)
    sel = torch.full((n + 2,), GUARD, device="cuda", dtype=torch.float64)
    _lib.check(_lib.lib().mk_integrate_final(s0.data_ptr(), n, N, 40.0, 1e-2, 0.9, K.data_ptr(), last.data_ptr(),
                                             sel.data_ptr(), None))
    return K.cpu().numpy(), last.cpu().numpy(), sel.cpu().numpy()


def _history(s0, T, N):
    n = len(s0)
    S = torch.full((T * n + 2, 8), GUARD, device="cuda", dtype=torch.float64)
    D = torch.full((T * n + 2,), GUARD, device="cuda", dtype=torch.float64)
    _lib.check(_lib.lib().mk_integrate_history(s0.data_ptr(), n, N, 40.0, 1e-2, 0.9, T, S.data_ptr(), D.data_ptr(), None))
    return S.cpu().numpy(), D.cpu().numpy()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 130])
@pytest.mark.parametrize("N", [1, 2, 301, 2500])
def test_walks_of_ragged_counts(n, N):
    s0 = _start(n)
    K, last, sel = _final(s0, N)
    assert np.all(K[n:] == -7) and np.all(last[n:] == GUARD) and np.all(sel[n:] == GUARD)
    K1, last1, sel1 = (np.concatenate(x) for x in zip(*[[a[:1] for a in _final(s0[p:p + 1].contiguous(), N)]
                                                        for p in range(n)]))
    np.testing.assert_array_equal(K[:n], K1)
    np.testing.assert_array_equal(last[:n], last1)
    np.testing.assert_array_equal(sel[:n], sel1)
    T = min(N, 700)  # rays end before and after the last row
    S, D = _history(s0, T, N)
    assert np.all(S[T * n:] == GUARD) and np.all(D[T * n:] == GUARD)
    S, D = S[:T * n].reshape(T, n, 8), D[:T * n].reshape(T, n)
    np.testing.assert_array_equal((D != 0).sum(0), np.minimum(K[:n], T))
    ended = K[:n] < T
    np.testing.assert_array_equal(S[-1][ended], last[:n][ended])
    if T == N:
        np.testing.assert_array_equal(S[-1], last[:n])
    for p in (0, n - 1):
        S1, D1 = _history(s0[p:p + 1].contiguous(), T, N)
        np.testing.assert_array_equal(S[:, p], S1[:T])
        np.testing.assert_array_equal(D[:, p], D1[:T])


@pytest.mark.parametrize("spin,inc", [(0.9, 85.0), (-0.9, 20.0), (0.94, 85.0), (0.95, 60.0), (0.98, 85.0), (0.0, 45.0)])
@pytest.mark.parametrize("n", [1, 3, 1023, 1024, 1025, 2001])
def test_bisection_schedules_give_the_sequential_radii(spin, inc, n, monkeypatch):
    ang = np.arange(n) / n * 2 * np.pi + 0.1
    got = ma.find_shadow_bisection_angles(spin, inc, ang)
    monkeypatch.setenv("MK_BISECT_BAND", "0")  # tree rounds
    np.testing.assert_array_equal(got, ma.find_shadow_bisection_angles(spin, inc, ang))
    few = slice(0, None, max(1, n // 3))
    np.testing.assert_array_equal(got[few], c_oracle.find_shadow_bisection_angles(spin, inc, ang[few], 2000, 1e-3, 40,
                                                                                  distance=1000.0))


@pytest.mark.parametrize("n", [1, 63, 65])
@pytest.mark.parametrize("N", [1, 2, 301, 2500])
def test_history_in_one_walk_equals_two(n, N):
    """geodesic_integrator finds T on the way when N rows are small: the rows
    and T are those of the walk that finds T and the walk that writes."""
    s0 = _start(n).cpu().numpy()
    s0[n // 2, 1:4] *= 10.0  # starts beyond 1500 M: frozen from row 0
    S, D = ma.geodesic_integrator(N, s0, 40, 1e-2, 0.9)
    S2, D2 = ma.geodesic_integrator(N, s0, 40, 1e-2, 0.9, max_chunk_bytes=1)  # one ray at a time
    np.testing.assert_array_equal(np.asarray(S), np.asarray(S2))
    np.testing.assert_array_equal(np.asarray(D), np.asarray(D2))


def test_history_in_one_walk_of_rays_that_are_all_frozen():
    s0 = _start(65).cpu().numpy()
    s0[:, 1:4] *= 10.0
    S, D = ma.geodesic_integrator(7, s0, 40, 1e-2, 0.9)
    S2, D2 = ma.geodesic_integrator(7, s0, 40, 1e-2, 0.9, max_chunk_bytes=1)
    np.testing.assert_array_equal(np.asarray(S), np.asarray(S2))
    np.testing.assert_array_equal(np.asarray(D), np.asarray(D2))
    assert not np.asarray(D).any()


def test_history_in_one_walk_is_complete_on_return():
    """mk_integrate_rows synchronises its stream: on return the rows behind each
    ray's last one are written too, also on a stream that no other waits for."""
    n, N = 50000, 400
    s0 = _start(144)[torch.arange(n, device="cuda") % 144].contiguous()
    s0[:, 1:4] *= 10.0  # beyond 1500 M: frozen from row 0, all their rows repeat
    s0[7] = _start(8)[7]
    S = torch.full((N, n, 8), GUARD, device="cuda", dtype=torch.float64)
    D = torch.full((N, n), GUARD, device="cuda", dtype=torch.float64)
    K = torch.empty(n, device="cuda", dtype=torch.int32)
    T = C.c_long()
    torch.cuda.synchronize()
    st = torch.cuda.Stream()
    _lib.check(_lib.lib().mk_integrate_rows(s0.data_ptr(), n, N, 40.0, 1e-2, 0.9, S.data_ptr(), D.data_ptr(),
                                            K.data_ptr(), C.byref(T), st.cuda_stream))
    done = st.query()
    with torch.cuda.stream(torch.cuda.Stream()):
        rest = S[T.value - 1].cpu()
    assert done
    st.synchronize()
    rows = torch.arange(n) != 7
    assert torch.equal(rest[rows], s0.cpu()[rows]) and not D[:T.value].cpu()[:, rows].any()


@pytest.mark.parametrize("spin,inc", [(0.0, 10.0), (0.5, 30.0), (0.97, 80.0)])
@pytest.mark.parametrize("n", [1, 65, 1025])
def test_bisection_to_small_errors(spin, inc, n, monkeypatch):
    """More halvings than the band's width is first searched for."""
    ang = np.arange(n) / n * 2 * np.pi + 0.1
    for err, it in ((1e-6, 40), (1e-9, 40), (0.0, 20)):
        got = ma.find_shadow_bisection_angles(spin, inc, ang, error_allowed=err, max_it=it)
        with monkeypatch.context() as mp:
            mp.setenv("MK_BISECT_BAND", "0")  # tree rounds
            np.testing.assert_array_equal(got, ma.find_shadow_bisection_angles(spin, inc, ang, error_allowed=err, max_it=it))
