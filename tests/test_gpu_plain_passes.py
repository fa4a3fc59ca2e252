"""Passes above norb 12 that run on the plain fiber kernel (few electrons, few
columns), and every way a diagonal evolution is applied inside a sequence: fused
into a pipelined or a plain pass, or by itself after the rotation."""

import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ffsim_amd
from ffsim_amd import _lib
from oracle import oracle as O

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]

# eps times the square root of the rotations per amplitude, on normalized states
TOL = {"complex128": 1e-12, "complex64": 2e-5}
DTYPES = ["complex128", "complex64"]
# tests/test_pass_rules_host.py holds the rule to these
PLAIN = [(17, (2, 3)), (18, (3, 3)), (16, (1, 8)), (18, (0, 3)), (18, (3, 18))]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("norb,nelec", PLAIN + [(18, (3, 4)), (17, (3, 5))])
def test_rotation_of_product_states(norb, nelec, dtype):
    rng = np.random.default_rng(norb * 100 + nelec[1])
    facs = [O.random_state_vector(ffsim_amd.dim(norb, n), rng) for n in nelec]
    mats = [ffsim_amd.random.random_unitary(norb, seed=rng) for _ in nelec]
    state = torch.from_numpy(np.kron(*facs).astype(dtype)).cuda()
    for pair in ((mats[0], mats[1]), (None, mats[1]), (mats[0], None)):
        got = ffsim_amd.apply_orbital_rotation(state, pair, norb, nelec).cpu().numpy()
        want = np.kron(*[f if m is None else O.apply_orbital_rotation(f, m, norb, n)
                         for f, m, n in zip(facs, pair, nelec)])
        bound = TOL[dtype] * (1.0 if dtype == "complex128" else np.abs(want).max())
        assert np.abs(got - want).max() <= bound


def _diagonal_launches(f):
    out = (ctypes.c_double * 6)()
    _lib.call("ffsim_amd_profile_begin")
    f()
    _lib.call("ffsim_amd_profile_end", out)
    return int(out[4])


@pytest.mark.parametrize("norb,nelec,dtype,separate", [
    # both last passes plain
    (17, (2, 3), "complex128", 0), (17, (2, 3), "complex64", 0), (18, (3, 3), "complex128", 0),
    (15, (3, 0), "complex64", 0),
    # alpha plain, beta pipelined over windows: the plain fused store in complex128
    (17, (4, 5), "complex128", 0), (17, (3, 8), "complex128", 0), (17, (3, 5), "complex64", None),
    # both pipelined
    (16, (5, 6), "complex128", 0), (16, (3, 8), "complex64", 0), (14, (7, 2), "complex64", 0),
    # whole beta sectors whose fused tile exceeds the LDS
    (15, (7, 3), "complex64", 2), (16, (2, 14), "complex64", 2),
])
def test_ansatz_equals_its_gates(norb, nelec, dtype, separate):
    rng = np.random.default_rng(norb + nelec[1])
    n_reps = 2
    rots = np.stack([ffsim_amd.random.random_unitary(norb, seed=rng) for _ in range(n_reps)])
    mats = rng.uniform(-3, 3, (n_reps, 2, norb, norb))
    mats = mats + mats.transpose(0, 1, 3, 2)
    op = ffsim_amd.UCJOpSpinBalanced(diag_coulomb_mats=mats, orbital_rotations=rots)
    g = torch.Generator(device="cuda").manual_seed(3)
    state = torch.empty(ffsim_amd.dim(norb, nelec), dtype=getattr(torch, dtype), device="cuda")
    torch.view_as_real(state).normal_(generator=g)
    state /= torch.linalg.vector_norm(state)
    got = state.clone()

    def run():
        ffsim_amd.apply_unitary(got, op, norb, nelec, copy=False)

    n = _diagonal_launches(run)
    if separate is not None:
        assert n == separate
    want = state.clone()
    for (aa, ab), u in zip(mats, rots):
        want = ffsim_amd.apply_diag_coulomb_evolution(want, (aa, ab, aa), -1.0, norb, nelec,
                                                      orbital_rotation=u)
    err = (got - want).abs().max().item()
    assert err <= TOL[dtype] * (1.0 if dtype == "complex128" else want.abs().max().item())
