"""Rotations of small states whose one sector is empty or full: a single row or
column, alone and in batches, on states with one element between them."""

import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ffsim_amd
from ffsim_amd import _lib
from ffsim_amd.gates.orbital_rotation import orbital_rotations_in_place
from oracle import oracle as O

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]

# eps times the square root of the rotations per amplitude, on normalized states
TOL = {"complex128": 1e-12, "complex64": 2e-5}


def _launches(f):
    out = (ctypes.c_double * 6)()
    _lib.call("ffsim_amd_profile_begin")
    f()
    _lib.call("ffsim_amd_profile_end", out)
    return int(out[1])


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n_states", [1, 3, 40])
@pytest.mark.parametrize("norb,nelec", [(6, (0, 0)), (6, (6, 2)), (7, (3, 0)), (10, (0, 5)),
                                        (11, (5, 11)), (12, (6, 0)), (12, (12, 6)), (12, (1, 12))])
def test_single_row_or_column(norb, nelec, n_states, dtype):
    rng = np.random.default_rng(norb * 1000 + n_states)
    dim = ffsim_amd.dim(norb, nelec)
    facs = [O.random_state_vector(ffsim_amd.dim(norb, n), rng) for n in nelec]
    buf = torch.full((n_states * (dim + 1) + 1,), 7.0, dtype=getattr(torch, dtype), device="cuda")
    states = [buf[1 + i * (dim + 1):][:dim] for i in range(n_states)]
    start = torch.from_numpy(np.kron(*facs).astype(dtype)).cuda()
    mats = [tuple(ffsim_amd.random.random_unitary(norb, seed=rng) for _ in nelec)
            for _ in range(n_states)]
    for s in states:
        s.copy_(start)
    n = _launches(lambda: orbital_rotations_in_place(states, mats, norb, nelec))
    # one launch per sector, however many the states
    assert n == 2
    assert torch.all(buf[:: dim + 1] == 7.0)
    for i in {0, n_states // 2, n_states - 1}:
        want = np.kron(*[O.apply_orbital_rotation(f, m, norb, k)
                         for f, m, k in zip(facs, mats[i], nelec)])
        bound = TOL[dtype] * (1.0 if dtype == "complex128" else np.abs(want).max())
        assert np.abs(states[i].cpu().numpy() - want).max() <= bound
        # the state alone: the same bits
        alone = start.clone()
        ffsim_amd.apply_orbital_rotation(alone, mats[i], norb, nelec, copy=False)
        assert torch.equal(alone, states[i])
