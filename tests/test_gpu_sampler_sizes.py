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
