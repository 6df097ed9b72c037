"""The sampler's launches by size (grmhd/athenak.py:618-812 of the reference):
each sample's scalars are the same bits whatever launch it is part of, and
nothing is written past the last."""
import numpy as np
import pytest
import torch

from mahakala_amd import _lib
from mahakala_amd.grmhd import synthetic as syn
from mahakala_amd.grmhd.athenak import AthenakFluidModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 257, 1499999, 1500000, 2999999, 3000000 + 17])
def test_scalars_do_not_depend_on_the_launch(n):
    m = AthenakFluidModel.from_datasets(syn.uniform_torus_snapshot(0.9, seed=0), 0.9, fluid_gamma=13. / 9)
    base = 4096
    g = torch.Generator(device="cuda").manual_seed(1)
    S = torch.empty((base, 8), device="cuda", dtype=torch.float64).uniform_(-1, 1, generator=g)
    S[:, 1:4] *= 30.0  # some outside the domain's inner blocks, some inside the horizon
    S[:, 4] -= 2.0
    lib = _lib.lib()

    def sample(states):
        k = len(states)
        out = torch.full((5 * k + 3,), -7.0, device="cuda", dtype=torch.float64)
        _lib.check(lib.mk_sample_scalars(m.device_snapshot.handle, states.data_ptr(), k, 0.9, np.pi / 3, out.data_ptr(),
                                         None))
        assert (out[5 * k:] == -7.0).all()
        return out[:5 * k].reshape(5, k)

    idx = torch.arange(n, device="cuda") % base
    got, ref = sample(S[idx].contiguous()), sample(S)[:, idx]
    assert torch.equal(got.view(torch.int64), ref.contiguous().view(torch.int64))


def test_pitch_of_momenta_orthogonal_to_the_flow():
    """k.u = 0 exactly (k^t = 0 in a flow at rest in the normal frame): the cosine
    k.b / (|k.u| |b|) is infinite and clamped to +-1; the fallback angle is for
    0/0 only, k.b = 0 or b = 0 (athenak.py:787-793)."""
    ds = syn.torus_snapshot(0.0, nblocks=2, n=8)
    ds["uov"][1:4] = 0.0
    ds["B"][:] = 0.0
    ds["B"][0] = 1.0
    ds["B"][:, 0] = 0.0  # no field in the first block
    m = AthenakFluidModel.from_datasets(ds, 0.0, fluid_gamma=13. / 9)
    rng = np.random.Generator(np.random.PCG64(2))
    S = np.zeros((400, 8))
    S[:, 1:4] = rng.uniform(-30, 30, (400, 3))
    S[:, 5] = rng.uniform(0.1, 1.0, 400) * np.where(rng.uniform(size=400) < 0.5, -1, 1)
    S[::5, 5] = 0.0  # k = 0
    sc = m.get_fluid_scalars_from_geodesics(S[None])
    assert not np.asarray(sc["kdotu"]).any()
    b, pitch = np.asarray(sc["b"])[0], np.asarray(sc["pitch_angle"])[0]
    assert 0 < (b == 0).sum() < 400
    want = np.where((b == 0) | (S[:, 5] == 0), np.arccos(np.cos(np.pi / 3)), np.where(S[:, 5] > 0, 0.0, np.pi))
    np.testing.assert_allclose(pitch, want, rtol=0, atol=4e-16)


@pytest.mark.parametrize("n", [5999999, 6000000 + 65])
def test_scalars_around_the_streamed_stores(n):
    test_scalars_do_not_depend_on_the_launch(n)
