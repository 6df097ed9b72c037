"""The transfer scans' tile kernels against the kernels of one thread per ray
(transfer.py:89-144 of the reference): the same bits for the same ray, at the
edges of the 64-row tiles and 16-ray blocks."""
import numpy as np
import pytest
import torch

from mahakala_amd import _lib, transfer

pytestmark = pytest.mark.gpu
MANY = 32768 + 17  # beyond the tile kernels' range


@pytest.mark.parametrize("T", [1, 2, 3, 64, 65, 66, 129, 193])
def test_tile_scans_equal_one_thread_per_ray(T):
    rng = np.random.Generator(np.random.PCG64(T))
    j, al = rng.exponential(1.0, (2, T, MANY))
    dt = -rng.exponential(0.1, (T, MANY))
    dt[T // 2:, ::3] = 0.0  # frozen rows
    j[0, 5], al[-1, 7] = np.nan, np.inf
    I, dI = transfer.solve_specific_intensity(j, al, dt, 0.5, dIs=True)
    att = transfer.solve_attenuated_emissivity(j, al, dt, 0.5)
    for n in (1, 15, 16, 17, 300):
        a = [np.ascontiguousarray(v[:, :n]) for v in (j, al, dt)]
        np.testing.assert_array_equal(transfer.solve_specific_intensity(*a, 0.5), I[:n])
        In, dIn = transfer.solve_specific_intensity(*a, 0.5, dIs=True)
        np.testing.assert_array_equal(In, I[:n])
        np.testing.assert_array_equal(dIn, dI[:, :n])
        np.testing.assert_array_equal(transfer.solve_attenuated_emissivity(*a, 0.5), att[:, :n])
    ref = np.zeros(MANY)
    with np.errstate(invalid="ignore"):
        for i in range(T - 1, 0, -1):
            ref = ref - dt[i - 1] * 0.5 * (j[i] - al[i] * ref)
    np.testing.assert_allclose(I, ref, rtol=1e-12)


@pytest.mark.parametrize("T", [2, 3, 5, 17, 64, 65, 66, 129, 130, 300])
def test_infinite_intensities_stay_infinite(T):
    """Intensities that become infinite in the row nearest the camera, with T - 1
    on and off a multiple of the tile: no row behind the last one is added."""
    rng = np.random.Generator(np.random.PCG64(T))
    j, al = rng.exponential(1.0, (2, T, MANY))
    dt = -rng.exponential(0.1, (T, MANY))
    j[1, 1], j[1, 2] = np.inf, -np.inf
    j[1, 3], dt[0, 3] = 1e308, -100.0  # overflows
    j[1, 4], dt[0, 4] = np.inf, 0.0    # 0 * inf: NaN in the reference too
    I, dI = transfer.solve_specific_intensity(j, al, dt, 0.5, dIs=True)
    ref = np.zeros(MANY)
    with np.errstate(invalid="ignore", over="ignore"):
        for i in range(T - 1, 0, -1):
            ref = ref - dt[i - 1] * 0.5 * (j[i] - al[i] * ref)
    np.testing.assert_array_equal(ref[1:4], [np.inf, -np.inf, np.inf])
    np.testing.assert_array_equal(I[1:5], ref[1:5])
    for n in (5, 16, 33):
        a = [np.ascontiguousarray(v[:, :n]) for v in (j, al, dt)]
        np.testing.assert_array_equal(transfer.solve_specific_intensity(*a, 0.5), I[:n])
        In, dIn = transfer.solve_specific_intensity(*a, 0.5, dIs=True)
        np.testing.assert_array_equal(In, I[:n])
        np.testing.assert_array_equal(dIn, dI[:, :n])


@pytest.mark.parametrize("T", [32, 33, 64, 65])
def test_every_choice_of_kernel_gives_the_same_bits(T):
    """By rows, rays and whether a block's rays are one line of a row: numbers of
    rays on both sides of each limit, and arrays that start off a line."""
    n = 40000
    g = torch.Generator(device="cuda").manual_seed(T)
    j, al, dt = (torch.empty(T, n, device="cuda", dtype=torch.float64).exponential_(1.0, generator=g) for _ in range(3))
    dt *= -0.1

    def scan(v, shift=0):
        k = v[0].shape[1]
        p = []
        for x in v:  # copies at a byte offset of 8 * shift
            buf = torch.empty(T * k + shift, device="cuda", dtype=torch.float64)
            buf[shift:] = x.reshape(-1)
            p.append(buf[shift:])
        I = torch.empty(k, device="cuda", dtype=torch.float64)
        dI, att = torch.empty((2, T - 1, k), device="cuda", dtype=torch.float64)
        a = [x.data_ptr() for x in p]
        _lib.check(_lib.lib().mk_solve_intensity(*a, T, k, 0.5, I.data_ptr(), dI.data_ptr(), None))
        _lib.check(_lib.lib().mk_attenuated_emissivity(*a, T, k, 0.5, att.data_ptr(), None))
        torch.cuda.synchronize()
        return I, dI, att

    ref = scan([j, al, dt])
    for k, shift in [(16, 0), (17, 0), (12287, 0), (12288, 0), (12288, 1), (12289, 0), (12304, 0), (12304, 3), (16384, 0), (16385, 0),
                     (16400, 0), (32752, 0), (32768, 0), (32784, 0)]:
        got = scan([x[:, :k].contiguous() for x in (j, al, dt)], shift)
        for a, b in zip(got, ref):
            assert torch.equal(a, b[..., :k]), (k, shift)
