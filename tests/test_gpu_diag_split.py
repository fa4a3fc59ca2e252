"""Diagonal operators at the column splits of small states (256, 512, ... columns
a block, ragged last blocks, one to nine rows, several states) against the
oracle's energies."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ffsim_amd
from oracle import oracle as O

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]


@pytest.mark.parametrize("z_rep", [False, True])
@pytest.mark.parametrize("norb,nelec", [(1, (1, 0)), (9, (1, 4)), (11, (0, 4)), (12, (1, 6)),
                                        (12, (11, 5)), (13, (0, 6)), (12, (4, 6)), (14, (1, 7))])
def test_energies_and_phases(norb, nelec, z_rep):
    rng = np.random.default_rng(norb * 100 + nelec[0])
    mats = rng.uniform(-1, 1, (3, norb, norb))
    mats = tuple(m + m.T for m in mats)
    e = O.diag_coulomb_energies(mats, norb, nelec, z_representation=z_rep).reshape(-1)
    vec = O.random_state_vector(ffsim_amd.dim(norb, nelec), rng)
    state = torch.from_numpy(vec).cuda()
    got = ffsim_amd.apply_diag_coulomb_evolution(state, mats, 0.3, norb, nelec,
                                                 z_representation=z_rep).cpu().numpy()
    # rounding of E: eps times the terms' moduli (random signs keep the sum's own
    # roundings below that); of a phase also one product per factor
    eps, terms = 2.3e-16, sum(np.abs(m).sum() for m in mats)
    tol = eps * (2 * norb + 8 + 0.3 * terms) * np.abs(vec).max()
    assert np.abs(got - np.exp(-0.3j * e) * vec).max() <= tol
    op = ffsim_amd.contract.diag_coulomb_linop(mats, norb, nelec, z_representation=z_rep)
    got = (op @ state).cpu().numpy()
    tol = eps * (8 + terms) * np.abs(vec).max()
    assert np.abs(got - e * vec).max() <= tol
