"""Transition RDMs where the minors' 4 x 4 blocks are ragged (1 to 13 empty
orbitals), with 0 and norb electrons, few and many columns, against the oracle."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ffsim_amd
from ffsim_amd.variational.gradient import DeviceAdjointOps
from oracle import oracle as O

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("norb,nelec", [(1, (1, 0)), (1, (1, 1)), (4, (4, 1)), (5, (0, 3)),
                                        (7, (5, 2)), (8, (1, 8)), (10, (7, 3)), (13, (1, 2)),
                                        (12, (6, 5))])
def test_matches_oracle(norb, nelec, dtype):
    rng = np.random.default_rng(norb * 100 + nelec[0])
    dim = ffsim_amd.dim(norb, nelec)
    lam, psi = (O.random_state_vector(dim, rng).astype(dtype) for _ in range(2))
    ops = DeviceAdjointOps(norb, nelec)
    got = ops.host_rdm(ops.transition_rdm(torch.from_numpy(lam).cuda(),
                                          torch.from_numpy(psi).cuda()))
    want = O.transition_rdm(lam.astype(complex), psi.astype(complex), norb, nelec)
    # sums in double of products of rounded inputs, of normalized states
    np.testing.assert_allclose(got, want, atol=1e-14, rtol=0)
